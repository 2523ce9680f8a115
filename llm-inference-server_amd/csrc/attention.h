// Launch parameters shared by the paged-attention kernels (internal to libpagedkv).
#pragma once

#include "pkv_common.h"

namespace pkv {

struct AttnParams {
    void* out;
    int64_t out_st, out_sh;          // elements
    const void* q;
    int64_t q_st, q_sh;              // elements
    const void* k;
    const void* v;
    int64_t sb, ss, sh;              // pool strides (elements): block, slot, head
    int64_t num_blocks;
    int block_size, num_kv_heads, head_dim;
    const int64_t* tables;
    int64_t table_stride, table_width;
    const int64_t* ctx_lens;
    const int64_t* qsl;              // query_start_loc [num_seqs+1]; null => token i is seq i
    int num_seqs, num_heads, group;
    int64_t num_tokens;
    int max_query_len;
    float scale_log2;                // scale * log2(e): scores live in the base-2 domain
    float scale;                     // softmax scale, applied to the rounded dot product
    // split-KV decode workspace
    float* ws_o;                     // [num_seqs, num_heads, max_parts, head_dim]
    float* ws_ml;                    // [num_seqs, num_heads, max_parts, 2] = (max, denominator)
    int max_parts;
    // Split-KV merge counters, one per (sequence, KV head), zero between calls (null: too
    // many pairs). The one-launch decode kernel's last run of a (sequence, KV head) to
    // finish merges them all.
    uint32_t* ws_cnt;
    // Fused KV append (null = none). Decode: row seq of app_k / app_v
    // ([num_seqs, num_kv_heads, head_dim], element strides app_st, app_sh) goes to flat
    // pool slot app_slots[seq] and the attention sees it there. Prefill (MFMA kernel): row
    // t of [num_tokens, num_kv_heads, head_dim] goes to app_slots[t] and the kernel reads
    // the new positions from these rows.
    const void* app_k;
    const void* app_v;
    int64_t app_st, app_sh;
    const int64_t* app_slots;
    // log2(block_size) if it is a power of two, else -1.
    int block_shift;
    // Prefill MFMA kernel: contexts cut into at most `splits` even runs of at most
    // split_tiles 64-key tiles, partials in ws_o / ws_ml by (token, head, split); ws_rows
    // [num_tokens, num_heads] = splits the merge reads for a row (0: the row is finished;
    // null on decode batches). splits = 1: no workspace.
    int splits, split_tiles;
    int64_t split_items;               // workgroups that the splits of the batch make
    int* ws_rows;
    // Persistent MFMA decode: units (blocks x KV-head groups) before each sequence,
    // [num_seqs + 1], written by the decode kernel for its merge kernel.
    int* ws_pfx;
};

// Whether the byte offsets of rows 0 .. slots - 1 of a block fit the unsigned 32-bit per-lane
// offsets of the tuned kernels (a negative slot stride does not: the generic kernel's case).
inline bool slot_offsets_fit(const AttnParams& p, int slots, int itemsize) {
    return p.ss >= 0 && p.ss <= 0x7fffffff && (slots * p.ss + p.head_dim) * itemsize <= 0xffffffffll;
}

// One-launch MFMA decode (attn_decode_split.hip): whether it takes these parameters (with
// p.app_* set: including the fused append, whose source rows must be 16-byte aligned).
bool decode_split_applies(const AttnParams& p, int dtype);
int launch_decode_split(const AttnParams& p, int dtype, hipStream_t stream);
// The same kernel on fp32 prompts (p.qsl set, no fused append, p.max_parts sized for the
// table): 16 query rows a workgroup.
bool prompt_split_f32_applies(const AttnParams& p);
int launch_prompt_split_f32(const AttnParams& p, hipStream_t stream);
// Whether the batch's row tiles make at most two and a quarter rounds of the GPU there.
bool prompt_split_f32_few(const AttnParams& p);
// fp32 register kernel (attn_decode.hip): the shapes where it beats the kernel
// above; it appends nothing itself.
bool decode_f32_applies(const AttnParams& p);
int launch_decode_f32(const AttnParams& p, hipStream_t stream);
// True when launch_prefill_attention runs the MFMA kernel for these parameters (with
// p.app_* set: including the fused append, whose source rows must be 16-byte aligned).
bool prefill_tuned(const AttnParams& p, int dtype);

// How the prefill MFMA kernel cuts a batch's contexts (splits = 1: it does not), and the
// workspace that takes: runs of at most split_tiles 64-key tiles, at most `splits` of them
// per workgroup. From host copies of the lengths (qlen null: one token per sequence; ctx
// null: only max_context_len is known). The lengths only balance the launch: a longer
// context than told is attended to whole, in longer runs.
struct SplitPlan {
    int splits, split_tiles;
    int64_t items, rows_bytes, ml_bytes, o_bytes;
    int64_t total() const { return rows_bytes + ml_bytes + o_bytes; }
};
SplitPlan prefill_split_plan(int64_t num_seqs, int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                             int64_t num_tokens, const int64_t* ctx, const int64_t* qlen, int64_t max_context_len);
// Batches whose contexts are no longer than this are not split: the merge launch costs
// about what their few tiles take.
constexpr int64_t kSplitMinContext = 1024;

// Bytes reserved for the merge counters at the front of a decode workspace (a fixed
// size, so counters never overlap another call's partials in a reused workspace).
constexpr int64_t kMergeCounterBytes = 256 * 1024;

// Tokens per split-KV partial that the decode workspace holds: a run of a split context is
// never shorter.
constexpr int kDecodePart = 256;

// Persistent MFMA decode (attn_decode_mfma.hip): whether it takes a batch of these
// parameters (16-bit pools, block size 16, head_dim 64/128, GQA 1/2/4/8, a multiple of
// 4 KV heads, at most 1024 sequences, at least 512 MiB of K/V at the longest context),
// the floats its split-KV partials
// need (0 when it never applies to such sizes), and the launch (PKV_EUNSUPPORTED
// without an error when the device does not fit). It needs p.ws_pfx, p.ws_ml, p.ws_o.
constexpr int kDecodeMfmaMaxSeqs = 1024;
bool decode_mfma_applies(const AttnParams& p, int dtype, int64_t max_context_len);
bool decode_mfma_sizes_apply(int64_t num_seqs, int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                             int64_t max_context_len);
int64_t decode_mfma_partial_floats(int64_t num_kv_heads, int64_t group, int64_t head_dim);
int launch_decode_mfma(const AttnParams& p, int dtype, hipStream_t stream);

int launch_generic_attention(const AttnParams& p, int dtype, hipStream_t stream);
// fp32 pools, block size 16, head_dim 64/128, GQA 1/2/4/8, 16-byte aligned rows: the
// tiled fp32 kernel (any query lengths). Returns
// PKV_EUNSUPPORTED (without setting an error) for anything else.
int launch_f32_attention(const AttnParams& p, hipStream_t stream);
// fp32 pools, prefill / chunked-prefill batches (p.qsl set, no fused append, a row of at
// least 2 tokens), block size 16, head_dim 64/128, GQA 1/2/4/8, 16-byte aligned rows: the
// fp32 MFMA kernel. Returns PKV_EUNSUPPORTED (without setting an error) for anything else.
int launch_prefill_f32_mfma(const AttnParams& p, hipStream_t stream);
// Returns PKV_EUNSUPPORTED (without setting an error) when no tuned kernel matches.
int launch_prefill_attention(const AttnParams& p, int dtype, hipStream_t stream);

// ---- prefill dispatch order (the MFMA prefill kernels, 256-thread workgroups).
// A prefill grid walks (sequence slot, query block) items; sequence slot i runs the
// sequence with the i-th largest context (ties by index), so the workgroups with the
// longest causal ranges start first and the end of the launch is left to short ones
// (bf16 config 4 chunks: the occupancy drained over the last ~50 of ~345 us in index
// order; 314.2 -> 306.7 us per call). Ordering every (sequence, query block) pair
// longest first instead was slower (322-325 us): it scatters a sequence's query blocks,
// whose K/V tiles one L2 otherwise serves to all of them. Every workgroup ranks the
// batch's contexts itself (one load per sequence, replacing its own context and query
// start loads); batches of more than kPrefillSortSeqs sequences keep index order.
constexpr int kPrefillSortSeqs = 256;   // one sequence per thread

struct PrefillSeq {
    int seq;
    int64_t q_first;
    int q_len;
    int ctx;                            // context length clamped to the table width
};

// Called by every thread of a 256-thread workgroup (it holds two barriers).
__device__ __forceinline__ PrefillSeq prefill_seq(const AttnParams& p, int seq_slot, int block_size) {
    const int64_t cap = p.table_width * (int64_t)block_size;
    PrefillSeq r;
    if (p.num_seqs > kPrefillSortSeqs) {
        r.seq = seq_slot;
        r.q_first = p.qsl ? p.qsl[seq_slot] : seq_slot;
        r.q_len = p.qsl ? (int)(p.qsl[seq_slot + 1] - r.q_first) : 1;
        const int64_t c = p.ctx_lens[seq_slot];
        r.ctx = (int)(c < cap ? c : cap);
        return r;
    }
    __shared__ int s_ctx[kPrefillSortSeqs];
    __shared__ int s_order[kPrefillSortSeqs];
    __shared__ int64_t s_qsl[kPrefillSortSeqs + 1];
    const int t = (int)threadIdx.x;
    if (t < p.num_seqs) {
        const int64_t c = p.ctx_lens[t];
        s_ctx[t] = (int)(c < cap ? c : cap);
        s_qsl[t] = p.qsl ? p.qsl[t] : t;
    }
    if (t == 0) s_qsl[p.num_seqs] = p.qsl ? p.qsl[p.num_seqs] : p.num_seqs;
    __syncthreads();
    if (t < p.num_seqs) {
        const int ct = s_ctx[t];
        int rank = 0;
        for (int u = 0; u < p.num_seqs; ++u) {
            const int cu = s_ctx[u];
            rank += (cu > ct || (cu == ct && u < t)) ? 1 : 0;
        }
        s_order[rank] = t;
    }
    __syncthreads();
    r.seq = s_order[seq_slot];
    r.q_first = s_qsl[r.seq];
    r.q_len = (int)(s_qsl[r.seq + 1] - r.q_first);
    r.ctx = s_ctx[r.seq];
    return r;
}

// ---- work items of the 16-bit prefill kernel: (KV head, sequence, split, tile of ROWS
// query rows). Only items that exist are numbered (a sequence has ceil(q_len G / ROWS) row
// tiles, and as many splits as its context makes), from the lengths in device memory, so
// the grid holds no empty workgroups to speak of: with a (longest query, longest context)
// rectangle for every sequence, two thirds of a ragged batch's workgroups found nothing to
// do, held a slot (70 KiB of LDS) for ~2 us each and kept workgroups with work waiting
// (12 prompts of 8-61 tokens behind 0.6-7.5k: the last one started 43 us into the launch).
struct PrefillItem {
    int seq, kvh, split, row_tile;
    int q_len, ctx;                     // ctx clamped to the table width
    int splits;                         // of this launch: 1 if the grid cannot hold the splits
    int64_t q_first;
};

// Splits of a context of n_tiles key tiles: as few as runs of at most split_tiles make,
// never more than `splits`.
__device__ __forceinline__ int split_count(int n_tiles, int splits, int split_tiles) {
    if (splits < 2) return 1;
    const int n = (n_tiles + split_tiles - 1) / split_tiles;
    return n < 1 ? 1 : (n < splits ? n : splits);
}

// This workgroup's item (256 threads, all of them call it: it holds two barriers). False:
// none. The hardware hands workgroup L to XCD L % 8 and each XCD has its own L2: items are
// numbered row tile fastest, then split, then sequence (longest context first, as above),
// then KV head, and XCD x takes the x-th contiguous eighth, so the workgroups that re-read
// one sequence's K/V share an L2. Row tiles run last-first (the longest causal range first).
template <int ROWS, int KEYS>
__device__ __forceinline__ bool prefill_item(const AttnParams& p, int block_size, PrefillItem& r) {
    const int t = (int)threadIdx.x;
    const uint32_t G = (uint32_t)p.group;
    const int64_t cap = p.table_width * (int64_t)block_size;
    const uint32_t xcd = blockIdx.x % 8, at = blockIdx.x / 8;
    if (p.num_seqs > kPrefillSortSeqs) {
        // Index order over the full rectangle, never split.
        const uint32_t n_qb = ((uint32_t)p.max_query_len * G + ROWS - 1) / ROWS;
        const uint32_t per_head = n_qb * (uint32_t)p.num_seqs;
        const uint32_t n_items = per_head * (uint32_t)p.num_kv_heads;
        const uint32_t item = xcd * ((n_items + 7) / 8) + at;
        if (at >= (n_items + 7) / 8 || item >= n_items) return false;
        r.kvh = (int)(item / per_head);
        r.seq = (int)(item % per_head / n_qb);
        r.row_tile = (int)(n_qb - 1 - item % n_qb);
        r.split = 0;
        r.splits = 1;
        r.q_first = p.qsl ? p.qsl[r.seq] : r.seq;
        r.q_len = p.qsl ? (int)(p.qsl[r.seq + 1] - r.q_first) : 1;
        const int64_t c = p.ctx_lens[r.seq];
        r.ctx = (int)(c < cap ? c : cap);
        return r.row_tile * ROWS < r.q_len * (int)G;
    }
    __shared__ int s_ctx[kPrefillSortSeqs];
    __shared__ uint32_t s_tiles[kPrefillSortSeqs];   // row tiles
    __shared__ uint32_t s_items[kPrefillSortSeqs];   // row tiles x splits
    __shared__ PrefillItem s_pick;
    __shared__ int s_found;
    int64_t q_first = 0;
    int q_len = 0, ctx = 0;
    uint32_t tiles = 0, items = 0;
    if (t < p.num_seqs) {
        const int64_t c = p.ctx_lens[t];
        q_first = p.qsl ? p.qsl[t] : t;
        q_len = p.qsl ? (int)(p.qsl[t + 1] - q_first) : 1;
        ctx = (int)(c < cap ? c : cap);
        tiles = q_len > 0 ? ((uint32_t)q_len * G + ROWS - 1) / ROWS : 0;
        items = tiles * (uint32_t)split_count((ctx + KEYS - 1) / KEYS, p.splits, p.split_tiles);
        s_ctx[t] = ctx;
        s_tiles[t] = tiles;
        s_items[t] = items;
    }
    if (t == 0) s_found = 0;
    __syncthreads();
    if (t < p.num_seqs) {
        uint32_t before = 0, total = 0, tiles_before = 0, tiles_total = 0;
        for (int u = 0; u < p.num_seqs; ++u) {
            const int cu = s_ctx[u];
            const bool first = cu > ctx || (cu == ctx && u < t);
            total += s_items[u];
            tiles_total += s_tiles[u];
            before += first ? s_items[u] : 0;
            tiles_before += first ? s_tiles[u] : 0;
        }
        int splits = p.splits;
        if (splits > 1 && (total * (uint32_t)p.num_kv_heads + 7) / 8 > gridDim.x / 8) {
            // Longer contexts than the grid was sized for: unsplit.
            splits = 1;
            total = tiles_total;
            before = tiles_before;
            items = tiles;
        }
        const uint32_t n_items = total * (uint32_t)p.num_kv_heads;
        const uint32_t item = xcd * ((n_items + 7) / 8) + at;
        if (at < (n_items + 7) / 8 && item < n_items) {
            const uint32_t kvh = item / total;
            const uint32_t in_head = item - kvh * total;
            if (in_head >= before && in_head - before < items) {
                const uint32_t in_seq = in_head - before;
                const uint32_t split = in_seq / tiles;
                s_pick = PrefillItem{t, (int)kvh, (int)split, (int)(tiles - 1 - (in_seq - split * tiles)), q_len, ctx,
                                     splits, q_first};
                s_found = 1;
            }
        }
    }
    __syncthreads();
    if (!s_found) return false;
    // Uniform: into scalar registers.
    r.seq = __builtin_amdgcn_readfirstlane(s_pick.seq);
    r.kvh = __builtin_amdgcn_readfirstlane(s_pick.kvh);
    r.split = __builtin_amdgcn_readfirstlane(s_pick.split);
    r.row_tile = __builtin_amdgcn_readfirstlane(s_pick.row_tile);
    r.q_len = __builtin_amdgcn_readfirstlane(s_pick.q_len);
    r.ctx = __builtin_amdgcn_readfirstlane(s_pick.ctx);
    r.splits = __builtin_amdgcn_readfirstlane(s_pick.splits);
    r.q_first = readlane64(s_pick.q_first, 0);
    return true;
}

}  // namespace pkv
