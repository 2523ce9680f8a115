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
// above; and whether it takes the fused append of p.app_* (16-byte source rows, small batches).
bool decode_f32_applies(const AttnParams& p);
bool decode_f32_appends(const AttnParams& p);
int launch_decode_f32(const AttnParams& p, hipStream_t stream);
// True when launch_prefill_attention runs the MFMA kernel for these parameters (with
// p.app_* set: including the fused append, whose source rows must be 16-byte aligned).
bool prefill_tuned(const AttnParams& p, int dtype);
// What it asks of the shape alone.
bool prefill_shape(int64_t block_size, int64_t head_dim, int dtype);

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
constexpr int kPrefillWaveSeqs = 16;

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

// This workgroup's item (256 threads, all of them call it: it may hold two barriers). False:
// none. The hardware hands workgroup L to XCD L % 8 and each XCD has its own L2: items are
// numbered row tile fastest, then split, then sequence (longest context first, as above),
// then KV head, and XCD x takes the x-th contiguous eighth, so the workgroups that re-read
// one sequence's K/V share an L2. Row tiles run last-first (the longest causal range first).
// Every workgroup pays for this search before its first load, so it takes one LDS read a
// sequence, in the waves that hold sequences only, and none in batches of up to 16 (three
// reads a sequence before: 200 prompts of 1-8 tokens behind up to 500, 12 heads of 64, fp16,
// 67 -> 52 us a call; 200 of 1-30 behind up to 200 55 -> 39; 8 of 16-500 17.4 -> 16.3).
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
    // Small batches: every wave for itself, without LDS or a barrier.
    const bool in_wave = p.num_seqs <= kPrefillWaveSeqs;
    const int lane = t & 63, s = in_wave ? lane : t;
    int64_t q_first = 0;
    int q_len = 0, ctx = 0, key = -1;
    uint32_t tiles = 0, items = 0;
    if (s < p.num_seqs) {
        const int64_t c = p.ctx_lens[s];
        q_first = p.qsl ? p.qsl[s] : s;
        q_len = p.qsl ? (int)(p.qsl[s + 1] - q_first) : 1;
        ctx = (int)(c < cap ? c : cap);
        tiles = q_len > 0 ? ((uint32_t)q_len * G + ROWS - 1) / ROWS : 0;
        items = tiles * (uint32_t)split_count((ctx + KEYS - 1) / KEYS, p.splits, p.split_tiles);
        // Longest context first, ties by index (contexts of 2^23 tokens count as tied).
        const int k = ctx < 0 ? 0 : ctx < (1 << 23) ? ctx : (1 << 23) - 1;
        key = k << 8 | (255 - s);
    }
    uint32_t before = 0, total = 0, tiles_before = 0, tiles_total = 0;
    const bool cut = p.splits > 1;            // else a row tile is an item
    if (in_wave) {
        for (int u = 0; u < p.num_seqs; ++u) {
            const bool first = __builtin_amdgcn_readlane(key, u) > key;
            const uint32_t iu = (uint32_t)__builtin_amdgcn_readlane((int)items, u);
            total += iu;
            before += first ? iu : 0;
            if (cut) {
                const uint32_t tu = (uint32_t)__builtin_amdgcn_readlane((int)tiles, u);
                tiles_total += tu;
                tiles_before += first ? tu : 0;
            }
        }
    }
    // Whether this workgroup's item is the sequence's; then r is its item (but seq, q_len, ctx
    // and q_first).
    auto mine = [&]() {
        r.splits = p.splits;
        if (cut && (total * (uint32_t)p.num_kv_heads + 7) / 8 > gridDim.x / 8) {
            // Longer contexts than the grid was sized for: unsplit.
            r.splits = 1;
            total = tiles_total;
            before = tiles_before;
            items = tiles;
        }
        const uint32_t n_items = total * (uint32_t)p.num_kv_heads;
        const uint32_t item = xcd * ((n_items + 7) / 8) + at;
        if (at >= (n_items + 7) / 8 || item >= n_items) return false;
        const uint32_t kvh = item / total;
        const uint32_t in_seq = item - kvh * total - before;     // wraps below the sequence's first
        if (in_seq >= items) return false;
        r.kvh = (int)kvh;
        r.split = (int)(in_seq / tiles);
        r.row_tile = (int)(tiles - 1 - in_seq % tiles);
        return true;
    };
    bool found;
    if (in_wave) {
        const uint64_t lanes = __builtin_amdgcn_ballot_w64(mine());
        found = lanes != 0;
        const int src = found ? __builtin_ctzll(lanes) : 0;
        r = PrefillItem{src,
                        __builtin_amdgcn_readlane(r.kvh, src),
                        __builtin_amdgcn_readlane(r.split, src),
                        __builtin_amdgcn_readlane(r.row_tile, src),
                        __builtin_amdgcn_readlane(q_len, src),
                        __builtin_amdgcn_readlane(ctx, src),
                        __builtin_amdgcn_readlane(r.splits, src),
                        readlane64(q_first, src)};
    } else {
        __shared__ uint4 s_seq[kPrefillSortSeqs];   // one LDS read a step of the loop below
        __shared__ PrefillItem s_pick;
        __shared__ int s_found;
        if (t == 0) s_found = 0;
        if (t < p.num_seqs) s_seq[t] = make_uint4((uint32_t)key, items, tiles, 0u);
        __syncthreads();
        if (t < p.num_seqs) {
            if (cut) {
#pragma unroll 4
                for (int u = 0; u < p.num_seqs; ++u) {
                    const uint4 o = s_seq[u];
                    const bool first = (int)o.x > key;
                    total += o.y;
                    tiles_total += o.z;
                    before += first ? o.y : 0;
                    tiles_before += first ? o.z : 0;
                }
            } else {
#pragma unroll 4
                for (int u = 0; u < p.num_seqs; ++u) {
                    const uint2 o = *reinterpret_cast<const uint2*>(&s_seq[u]);
                    total += o.y;
                    before += (int)o.x > key ? o.y : 0;
                }
            }
            if (mine()) {
                s_pick = PrefillItem{t, r.kvh, r.split, r.row_tile, q_len, ctx, r.splits, q_first};
                s_found = 1;
            }
        }
        __syncthreads();
        found = s_found != 0;
        r = s_pick;
    }
    if (!__builtin_amdgcn_readfirstlane((int)found)) return false;
    // Uniform: into scalar registers.
    r.seq = __builtin_amdgcn_readfirstlane(r.seq);
    r.kvh = __builtin_amdgcn_readfirstlane(r.kvh);
    r.split = __builtin_amdgcn_readfirstlane(r.split);
    r.row_tile = __builtin_amdgcn_readfirstlane(r.row_tile);
    r.q_len = __builtin_amdgcn_readfirstlane(r.q_len);
    r.ctx = __builtin_amdgcn_readfirstlane(r.ctx);
    r.splits = __builtin_amdgcn_readfirstlane(r.splits);
    r.q_first = readlane64(r.q_first, 0);
    return true;
}

}  // namespace pkv
