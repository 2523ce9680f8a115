// Paged prefill / chunked-prefill attention on MFMA (gfx950), fp16/bf16, head_dim a
// multiple of 16 from 32 to 128, any GQA group, block sizes that are powers of two from 8
// up; decode batches whose shape the decode kernels do not take run here too (one query
// token per sequence). Other shapes take the generic kernel.
//
// Prefill is compute-bound (config 4 chunks: ~926 flop per byte touched), so the
// contraction runs on v_mfma_f32_32x32x16_{bf16,f16}. The formulation is chosen so
// the softmax needs almost no cross-lane traffic:
//
//  * S^T = K · Q^T per 32-key x 32-row tile: A = K rows (from LDS), B = Q^T
//    (registers, loaded once). MFMA result register r of lane l holds
//    S^T[key 8*(r/4) + 4*(l/32) + r%4][row l%32], so every lane owns ONE query row's
//    column: row max / row sum are lane-local over 32 values plus one permlane32 swap
//    with the lane holding the other half of the keys.
//  * P^T feeds the P·V MFMA as its B operand straight from the S^T accumulator
//    registers, cast to the pool dtype at the point where the reference casts
//    `probs.to(v.dtype)` — but as the unnormalised weights exp2(s - m) <= 2^8 of fp32
//    scores, divided by the fp32 row sum only at the end, where the reference rounds
//    its fp16 scores and then the normalised probabilities. The key order inside a
//    lane's 8 slots is the accumulator's, and the A operand V^T is read from LDS in that
//    same key order, so no data moves between the two MFMAs.
//  * V^T: the 64-key V tile is staged row-major like K and read through gfx950's
//    transposing LDS load (ds_read_b64_tr_b16): two 8-byte reads per MFMA give each
//    lane its 8 keys of one head_dim column.
//  * Work unit: one workgroup = (sequence, KV head, 128 query rows) x 4 waves of 32 rows.
//    A query row is one (token, query head of the KV head's group) pair, row f of a
//    sequence = token f / G, head f % G, so the rows of every group size (3 and 6
//    included) fill the tile and all share the staged K/V tiles: 64 keys walked through
//    the block table up to the causal bound of the workgroup's last token. A wave whose
//    own rows end before a tile skips its products and only stages.
//  * Split contexts: a batch of few query rows behind long contexts (cached prefixes,
//    chunks of a lone prompt, decode rows) makes too few workgroups to fill the GPU and
//    each walks its context serially, so the launch cuts the contexts into runs of
//    split_tiles tiles, one workgroup each, whose (max, denominator, unnormalised output)
//    go to the workspace in fp32 and are merged by prefill_merge_kernel. Measured, calls
//    through the Python entry: 12 prompts of 8-61 tokens behind 0.6-7.5k, 32/8 heads, bf16,
//    190 -> 72 us; decode of 24 sequences of up to 3k tokens, 24/8 heads, block size 32, fp16
//    (one wave per (token, head) before), 5,100 -> 38.6 us; 12 chunks of 24-190 tokens behind
//    up to 1.5k, 32 heads x 80, block size 32, bf16, 5,970 -> 62 us. prefill_split_plan
//    chooses.
//  * Two waves per SIMD (registers capped at 256 per lane): with one, every MFMA ->
//    softmax -> MFMA dependency and every load wait idles the matrix core; two
//    workgroups per CU interleave (config 4 chunks: 311 -> 486 TFLOP/s).
//  * XCD-aware order: the hardware hands workgroup L to XCD L % 8 and each XCD has its
//    own L2. Work items are numbered query block fastest, then split, then sequence, then
//    KV head, and XCD x takes the x-th contiguous eighth, so the workgroups that re-read
//    one sequence's K/V tiles share an L2 instead of fetching them from HBM once per XCD.
//    Within a sequence the query blocks go last-first (longest causal range first).
//  * Staging: K/V tiles move HBM -> LDS by DMA (global_load_lds_dwordx4), double
//    buffered: tile t+1 streams into one buffer pair while tile t is computed from the
//    other, one barrier per tile, no staging registers and no LDS store instructions.
//    A wave's whole-block DMA takes the block base as a uniform (scalar) base and a
//    fixed per-lane 32-bit offset, so an issue costs no vector address arithmetic (the
//    DMAs are inline asm, hidden from the compiler's wait counting: dma16); only
//    a block crossing the causal bound takes the per-row path. The LDS reads likewise
//    take per-lane offsets computed once and carry the buffer and key-group part as
//    immediates (config 4 chunks: 337 -> 328 us for the two together).
//    Rows are unpadded with an XOR swizzle of their 16-byte chunks (lds_swizzle), which
//    keeps the K and transposed V reads free of bank conflicts. The tile's block ids
//    come from one vector load issued a tile ahead, so no DMA waits on a table read.
//  * Block sizes: a wave stages 16 keys per tile as two 8-key halves, each inside one
//    block for any power of two >= 8. Block size 16 has instances of its own (one id per
//    wave and tile, no shifts).
//  * Online softmax in fp32, base-2 domain, with lazy rescaling (the running max is
//    raised only when a tile exceeds it by more than 2^8); causal mask key <= query
//    position, applied only on tiles that cross the workgroup's first query position,
//    with positions from context_lens - query_lens (reference core/attention.py:44-53).
//
// MFMA lane layouts (A, B, C of the 32x32x16 f16/bf16 forms) were pinned on the MI355X
// with a one-hot probe before this kernel was written.
#include "attention.h"

namespace pkv {
namespace {

constexpr int kBS = 16;
constexpr int kKT = 64;          // keys per staged tile
constexpr int kQT = 32;          // query rows per wave
constexpr int kRows = 4 * kQT;   // query rows per workgroup

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma;
template <>
struct Mfma<_Float16> {
    __device__ __forceinline__ static f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                      0, 0, 0);
    }
    __device__ __forceinline__ static uint32_t pack(float lo, float hi) {
        half2_t v = {(_Float16)lo, (_Float16)hi};
        return __builtin_bit_cast(uint32_t, v);
    }
};
template <>
struct Mfma<bf16_t> {
    __device__ __forceinline__ static f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                       c, 0, 0, 0);
    }
    __device__ __forceinline__ static uint32_t pack(float lo, float hi) {
        bf16x2_t v = {(__bf16)lo, (__bf16)hi};
        return __builtin_bit_cast(uint32_t, v);
    }
};

typedef short s16x4 __attribute__((ext_vector_type(4)));

// Transposing LDS read (gfx950 ds_read_b64_tr_b16). Within each group of 16 lanes the
// 16 source addresses name 4 consecutive 16-bit elements each; taking those 64
// elements in (lane, element) order, result lane i receives elements i, i+16, i+32
// and i+48. With source lane c of a group pointing at V[key0 + c/4][d0 + 4*(c%4)] of a
// row-major tile, lane i therefore receives V[key0 .. key0+3][d0 + i]: four keys of
// one head_dim column, the MFMA A-operand slice of V^T. (Semantics pinned on the
// MI355X with an in-bounds probe.)
__device__ __forceinline__ uint2 lds_read_tr16(const uint16_t* ptr) {
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4*)(ptr));
    return __builtin_bit_cast(uint2, v);
}

// XOR swizzle of a K/V tile row in LDS: logical 16-byte chunk c of row r sits in
// physical slot c ^ lds_swizzle<D>(r) of the unpadded row (period 16 rows). Two
// constraints, for 16- and 32-lane LDS passes alike:
//  * a b128 K read takes one logical chunk of 16 consecutive rows: the swizzle is a
//    permutation over any 16 aligned rows, so the 16 reads hit 16 distinct slots;
//  * 32 lanes of a transposing V read take 4 aligned rows x 4 consecutive logical
//    chunks (one aligned 4-chunk block): the 4 rows' swizzles move that block to 4
//    different blocks, so the 16 reads are distinct too.
// D = 128 (16 chunks = 256 bytes per row, one bank sweep): slot c ^ (4 (r % 4) + r / 4 % 4).
// D = 64 (8 chunks per 128-byte row, two rows per bank sweep): rows of one parity share
// the sweep half, so the same two rules apply to each parity: c ^ (4 bit1 + 2 bit2 + bit3).
// Other widths only meet the first rule: rows 4 apart start in the same banks at D = 32
// and 96 (c ^ r / 4 % 4), rows 8 apart at 48, 80 and 112 (c ^ r / 8 % 2).
template <int D>
__device__ __forceinline__ int lds_swizzle(int r) {
    if constexpr (D == 128) return ((r & 3) << 2) | ((r >> 2) & 3);
    else if constexpr (D == 64) return (((r >> 1) & 1) << 2) | (((r >> 2) & 1) << 1) | ((r >> 3) & 1);
    else if constexpr (D % 32 == 0) return (r >> 2) & 3;
    else return (r >> 3) & 1;
}

// Softmax maxima are only raised when a tile's max exceeds the running one by more
// than 2^8: until then probabilities are exp2(s - m) <= 256 (exact enough in fp32 and
// in the pool dtype), and the O accumulators need no rescale — FlashAttention-3's lazy
// rescaling, which removes the per-tile multiply of every accumulator.
constexpr float kRescaleThreshold = 8.f;

__device__ __forceinline__ uint32_t lds_u32(const void* p) {
    return (uint32_t)(uintptr_t)((const __attribute__((address_space(3))) char*)p);
}
// 16 bytes per lane by LDS DMA to LDS address lds + 16 lane (M0 = lds), from the uniform
// base sbase plus the lane's 32-bit offset, or from the lane's own 64-bit address. Issued
// from inline asm, so the compiler's wait counting never sees an LDS DMA in flight: with
// one in flight it cannot count LDS reads in order and waits for all of them (lgkmcnt(0))
// before every MFMA step (config 4 chunks: 314 -> 310 us). The tile's s_waitcnt(0) and
// barrier order the DMA's data for its readers. M0 is reserved to the compiler (a clobber
// of it is not honoured), so no compiler-generated code of this kernel may rely on M0:
// all of its LDS DMAs go through these helpers.
__device__ __forceinline__ void dma16(const char* sbase, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds), "v"(voff), "s"(sbase)
                 : "memory");
}
__device__ __forceinline__ void dma16(const char* addr, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(lds), "v"(addr)
                 : "memory");
}

// Tiles per split of a workgroup with n_tiles key tiles: its splits are of even lengths.
__device__ __forceinline__ int split_run(int n_tiles, int splits, int split_tiles) {
    const int n = split_count(n_tiles, splits, split_tiles);
    return (n_tiles + n - 1) / n;
}

template <typename T, int D, bool BS16>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void paged_prefill_kernel(
    const AttnParams p) {
    static_assert(D % 16 == 0 && D >= 32 && D <= 128, "head_dim");
    constexpr int DSTEPS = D / 16;            // QK^T contraction steps
    constexpr int DTILES = (D + 31) / 32;     // P·V output d tiles (the last may be half a tile)
    constexpr int ROWB = D * 2;               // bytes per K/V row
    constexpr int CPR = ROWB / 16;            // 16-byte chunks per row
    // DMA instructions (64 lanes x 16 B) per 16-row block, K or V; the last one is partly
    // masked where 16 rows are not whole instructions.
    constexpr int IPB = (kBS * CPR + 63) / 64;
    constexpr bool kWholeDma = kBS * CPR % 64 == 0;
    // Rows of one instruction all in one 8-row half of the block: the half's base is uniform.
    constexpr bool kHalfDma = 64 % CPR == 0 && 64 / CPR <= 8;

    // Two K/V tile buffers, distinct objects so the compiler can tell a DMA into one
    // from reads of the other (it waits on a pending LDS DMA only before reading the
    // buffer that DMA targets).
    __shared__ __attribute__((aligned(1024))) uint16_t s_k0[kKT * D];
    __shared__ __attribute__((aligned(1024))) uint16_t s_v0[kKT * D];
    __shared__ __attribute__((aligned(1024))) uint16_t s_k1[kKT * D];
    __shared__ __attribute__((aligned(1024))) uint16_t s_v1[kKT * D];

    // This workgroup's work item (prefill_item, attention.h).
    PrefillItem it;
    if (!prefill_item<kRows, kKT>(p, BS16 ? kBS : p.block_size, it)) return;
    const uint32_t G = (uint32_t)p.group;
    const int kvh = it.kvh, split = it.split, seq = it.seq;
    const int64_t q_first = it.q_first;
    const int q_len = it.q_len;
    const int ctx = it.ctx;
    const int n_rows = q_len * (int)G;        // query rows of the sequence
    const int row0 = it.row_tile * kRows;     // first row of this workgroup
    const int pos0 = ctx - q_len;             // position of query 0
    const int rows = n_rows - row0 < kRows ? n_rows - row0 : kRows;
    const int q0 = (int)((uint32_t)row0 / G);                    // first and last token of this workgroup
    const int q_last = (int)((uint32_t)(row0 + rows - 1) / G);
    const int kmax = pos0 + q_last + 1;       // keys [0, kmax) are visible to this workgroup
    if (kmax <= 0) return;
    const int first_pos = pos0 + q0;          // smallest query position in the workgroup
    // This workgroup's run of key tiles.
    const int n_tiles = (kmax + kKT - 1) / kKT;
    int t_begin = 0, t_end = n_tiles, run = n_tiles;
    if (it.splits > 1) {
        run = split_run(n_tiles, it.splits, p.split_tiles);
        t_begin = split * run;
        if (t_begin >= n_tiles) return;
        t_end = n_tiles - t_begin < run ? n_tiles : t_begin + run;
    }

    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int h = lane >> 5;                  // half of the wave
    const int col = lane & 31;                // query row of the wave / MFMA row-col index
    // This lane's query row: token my_q, head my_head of the group. Rows past the last one
    // repeat it (computed, not stored).
    const int wrow = wave * kQT + col;
    const bool my_live = wrow < rows;
    const uint32_t my_row = (uint32_t)(row0 + (my_live ? wrow : rows - 1));
    const int my_q = (int)(my_row / G);
    const int my_head = kvh * (int)G + (int)(my_row - (uint32_t)my_q * G);
    const int my_pos = pos0 + my_q;
    // Keys visible to this wave's rows (0: it has none, and only stages).
    const int wave_rows = rows - wave * kQT < kQT ? rows - wave * kQT : kQT;
    const int wave_kmax = wave_rows > 0 ? pos0 + (int)((uint32_t)(row0 + wave * kQT + wave_rows - 1) / G) + 1 : 0;

    f32x16 o[DTILES];
#pragma unroll
    for (int t = 0; t < DTILES; ++t) o[t] = f32x16{};
    float m_run = kNegInf, l_run = 0.f;       // running max (scaled, base 2) and denominator

    const int64_t* table = p.tables + (int64_t)seq * p.table_stride;
    const char* kbase = reinterpret_cast<const char*>(p.k) + (int64_t)kvh * p.sh * (int64_t)sizeof(T);
    const char* vbase = reinterpret_cast<const char*>(p.v) + (int64_t)kvh * p.sh * (int64_t)sizeof(T);
    const int64_t block_bytes = p.sb * (int64_t)sizeof(T);
    const int64_t slot_bytes = p.ss * (int64_t)sizeof(T);

    // Block ids of 64-key tile kt: lane l holds the block of the tile's 8-key half-group
    // l % 8 (block size 16: of its 16-key group l % 4), the index clamped to the last block
    // with a visible key, so every lane loads a valid table entry without a branch (kmax <=
    // context <= table width x block size). A group at or beyond kmax is staged by
    // position, never from its id: dma_tile sends it to the redirect path.
    const int nb_last = BS16 ? (kmax - 1) / kBS : (kmax - 1) >> p.block_shift;
    auto tile_ids = [&](int kt) -> int64_t {
        const int b = BS16 ? kt * (kKT / kBS) + (lane & 3) : (kt * kKT + 8 * (lane & 7)) >> p.block_shift;
        return table[b < nb_last ? b : nb_last];
    };
    // Tile staging by LDS DMA (global_load_lds_dwordx4: lane i's 16 bytes land at the
    // instruction's LDS base + 16 i, no registers involved). Wave w stages keys 16 w ..
    // 16 w + 15 of the tile for K and V; instruction j writes chunks 64 j .. 64 j + 63 of
    // those 16 rows. Rows at or beyond kmax, and blocks whose id is outside the pool, are
    // redirected to the tile's first row (a valid key): masked to -inf in S, so their
    // finite V rows get probability 0.
    // Row within the 16 and swizzled source chunk of this lane's instruction j.
    auto dma_row = [&](int j) { return (64 * j + lane) / CPR; };
    auto dma_chunk = [&](int j) { return (64 * j + lane) % CPR ^ lds_swizzle<D>((64 * j + lane) / CPR); };
    // This lane's byte offset inside an 8-row half (inside the block at block size 16) for
    // each of its DMA instructions, fixed for the whole kernel.
    uint32_t lane_off[IPB];
#pragma unroll
    for (int j = 0; j < IPB; ++j)
        lane_off[j] = (uint32_t)((BS16 ? dma_row(j) : dma_row(j) & 7) * slot_bytes) + (uint32_t)(dma_chunk(j) * 16);
    const bool offs_fit = kBS * slot_bytes + ROWB <= (int64_t)0xffffffff;
    const bool fused = p.app_k != nullptr;
    // With a fused append, key positions >= pos0 (this pass's new tokens) come from the
    // source rows: key position j is packed token q_first + j - pos0.
    const int new_from = fused ? pos0 : 0x7fffffff;
    const char* knew = fused ? reinterpret_cast<const char*>(p.app_k) + (int64_t)kvh * p.app_sh * (int64_t)sizeof(T)
                             : nullptr;
    const char* vnew = fused ? reinterpret_cast<const char*>(p.app_v) + (int64_t)kvh * p.app_sh * (int64_t)sizeof(T)
                             : nullptr;
    const int64_t new_row_bytes = p.app_st * (int64_t)sizeof(T);
    auto dma_tile = [&](int kt, int64_t ids, uint16_t* sk, uint16_t* sv) {
        const int row0 = kt * kKT + wave * kBS;                       // first key of this wave's group
        // Bytes from the pool head's base to the group's two 8-key halves.
        const int64_t id0 = readlane64(ids, 0);
        int64_t idw, idw2, half0, half1;
        if constexpr (BS16) {
            idw = idw2 = readlane64(ids, wave);
            half0 = idw * block_bytes;
            half1 = half0 + 8 * slot_bytes;
        } else {
            idw = readlane64(ids, 2 * wave);
            idw2 = readlane64(ids, 2 * wave + 1);
            half0 = idw * block_bytes + (row0 & (p.block_size - 1)) * slot_bytes;
            half1 = idw2 * block_bytes + ((row0 + 8) & (p.block_size - 1)) * slot_bytes;
        }
        const bool okw = ((uint64_t)idw < (uint64_t)p.num_blocks) & ((uint64_t)idw2 < (uint64_t)p.num_blocks);
        // The common case; one uniform branch (bitwise &: no short-circuit branches).
        if (okw & offs_fit & (row0 + kBS <= kmax) & (row0 + kBS <= new_from)) {
#pragma unroll
            for (int j = 0; j < IPB; ++j) {
                const int dst = wave * kBS * ROWB + j * 1024;
                if constexpr (BS16 && kWholeDma) {
                    dma16(kbase + half0, lane_off[j], lds_u32((char*)sk + dst));
                    dma16(vbase + half0, lane_off[j], lds_u32((char*)sv + dst));
                } else if constexpr (kHalfDma) {
                    const int64_t half = 64 * j / CPR < 8 ? half0 : half1;
                    dma16(kbase + half, lane_off[j], lds_u32((char*)sk + dst));
                    dma16(vbase + half, lane_off[j], lds_u32((char*)sv + dst));
                } else if (kWholeDma || 64 * j + lane < kBS * CPR) {
                    const int64_t off = (dma_row(j) < 8 ? half0 : half1) + lane_off[j];
                    dma16(kbase + off, lds_u32((char*)sk + dst));
                    dma16(vbase + off, lds_u32((char*)sv + dst));
                }
            }
            return;
        }
        // The redirect target, key kt * kKT: with a fused append it is a new row when it
        // lies at or past pos0 (its pool slot may be mid-write in this launch and its old
        // contents need not be finite, and a 0 probability times a NaN V is NaN).
        const int key0 = kt * kKT;
        const char* ksafe;
        const char* vsafe;
        if (key0 >= new_from) {
            const int64_t o = (q_first + key0 - pos0) * new_row_bytes;
            ksafe = knew + o;
            vsafe = vnew + o;
        } else {
            const int64_t o = (uint64_t)id0 < (uint64_t)p.num_blocks
                                  ? id0 * block_bytes + (BS16 ? 0 : (key0 & (p.block_size - 1)) * slot_bytes)
                                  : 0;
            ksafe = kbase + o;
            vsafe = vbase + o;
        }
#pragma unroll
        for (int j = 0; j < IPB; ++j) {
            const int r = dma_row(j);
            const int key = row0 + r;
            const int64_t chunk = (int64_t)(dma_chunk(j) * 16);
            const char* ks;
            const char* vs;
            if (key >= new_from && key < kmax) {                      // a new row: from the source
                const int64_t off = (q_first + key - pos0) * new_row_bytes + chunk;
                ks = knew + off;
                vs = vnew + off;
            } else if ((uint64_t)(r < 8 ? idw : idw2) < (uint64_t)p.num_blocks && key < kmax) {
                const int64_t off = (r < 8 ? half0 : half1) + (int64_t)(r & 7) * slot_bytes + chunk;
                ks = kbase + off;
                vs = vbase + off;
            } else {
                ks = ksafe + chunk;
                vs = vsafe + chunk;
            }
            const int dst = wave * kBS * ROWB + j * 1024;
            if (kWholeDma || 64 * j + lane < kBS * CPR) {
                dma16(ks, lds_u32((char*)sk + dst));
                dma16(vs, lds_u32((char*)sv + dst));
            }
        }
    };

    // Transposed V^T reads: source lane c of each 16-lane group points at key row
    // c / 4 of its 4-key group, head_dim column d0 + 4 * (c % 4); groups 0/2 cover
    // columns 0-15 of the 32-wide d tile, groups 1/3 columns 16-31.
    const int grp = lane >> 4;
    const int tr_key = (lane & 15) >> 2;
    const int tr_col = 16 * (grp & 1) + 4 * (lane & 3);

    // Swizzled LDS addresses (bytes) of this lane's operands. K: row half*32 + col,
    // logical chunk 2 s + h. V (transposing reads): rows kk + tr_key and kk + tr_key + 8
    // of the step's 16-key group kk, logical chunk (32 t + tr_col) / 8, 8-byte half
    // (lane & 1); the swizzle of those rows does not depend on the group.
    const int k_swz = lds_swizzle<D>(col);
    const int v_cb = (tr_col >> 3);
    const int v_lo_swz = lds_swizzle<D>(4 * (grp >> 1) + tr_key);
    const int v_hi_swz = lds_swizzle<D>(4 * (grp >> 1) + tr_key + 8);
    const int v_byte = 8 * (lane & 1);
    // Per-lane byte offsets inside a tile buffer, fixed for the kernel: the K read of
    // step s (row col) and the V^T reads of d tile t (rows tr_key, tr_key + 8 of a 16-key
    // group). Everything else in an LDS address — the buffer, the 32-key half, the key
    // group — is a constant the read instruction carries as its immediate offset.
    uint32_t koff[DSTEPS], voff_lo[DTILES], voff_hi[DTILES];
#pragma unroll
    for (int s = 0; s < DSTEPS; ++s) {
        koff[s] = (uint32_t)(col * ROWB + (((2 * s + h) ^ k_swz) << 4));
        asm volatile("" : "+v"(koff[s]));
    }
#pragma unroll
    for (int t = 0; t < DTILES; ++t) {
        // Columns past head_dim (the last tile of 48, 80, 112) re-read the tile's first
        // chunks: their products land in output rows that are never stored.
        const int c = 4 * t + v_cb < CPR ? 4 * t + v_cb : 4 * t + (v_cb & 1);
        voff_lo[t] = (uint32_t)((4 * (grp >> 1) + tr_key) * ROWB + v_byte + ((c ^ v_lo_swz) << 4));
        voff_hi[t] = (uint32_t)((4 * (grp >> 1) + tr_key + 8) * ROWB + v_byte + ((c ^ v_hi_swz) << 4));
        asm volatile("" : "+v"(voff_lo[t]), "+v"(voff_hi[t]));
    }

    // The first tile's block ids, then the queries, so that one memory round trip covers
    // both.
    int64_t ids = tile_ids(t_begin);
    // Q^T B operand: lane supplies Q[query my_q][d = 16*step + 8*h .. +8].
    u32x4 qfrag[DSTEPS];
    {
        const char* qrow = reinterpret_cast<const char*>(p.q) +
                           ((q_first + my_q) * p.q_st + (int64_t)my_head * p.q_sh) * (int64_t)sizeof(T);
#pragma unroll
        for (int s = 0; s < DSTEPS; ++s) {
            const Vec16 v = load16(qrow + (s * 16 + h * 8) * (int)sizeof(T));
            qfrag[s] = u32x4{v.w[0], v.w[1], v.w[2], v.w[3]};
        }
    }

    // Fused KV append (p.app_k set): the new K/V rows of the tokens whose first query row
    // is this workgroup's go to their pool slots (the first split writes them). Nothing in
    // this launch reads those slots: every workgroup stages positions >= pos0 from the
    // source rows instead (dma_tile), so no workgroup waits for another. It happens behind
    // the last tile: in front of the first one it held every workgroup up for 5.8 us (config 4
    // chunks), behind the first DMAs for 2.5-6 us (mixed chunks, 32 heads of 80: 47.2 -> 45.8
    // us a call for the move to the end; short tails 55.4 -> 54.2).
    constexpr int kAppend = 4;                // 16-byte pieces of K and V in flight per thread
    const int tok_begin = (int)(((uint32_t)row0 + G - 1) / G);
    const int n_pieces =
        fused && split == 0 ? ((int)(((uint32_t)(row0 + rows) + G - 1) / G) - tok_begin) * CPR : 0;
    Vec16 app_k[kAppend], app_v[kAppend];
    int64_t app_slot[kAppend];
    auto append_load = [&](int i0) {
#pragma unroll
        for (int j = 0; j < kAppend; ++j) {
            const int i = i0 + j * 256 + (int)threadIdx.x;
            app_slot[j] = -1;
            if (i < n_pieces) {
                const int64_t tok = q_first + tok_begin + i / CPR;
                const int64_t src = (tok * p.app_st + (int64_t)kvh * p.app_sh) * (int64_t)sizeof(T) + (i % CPR) * 16;
                app_slot[j] = p.app_slots[tok];
                app_k[j] = load16(reinterpret_cast<const char*>(p.app_k) + src);
                app_v[j] = load16(reinterpret_cast<const char*>(p.app_v) + src);
            }
        }
    };
    auto append_store = [&](int i0) {
        const int bs = BS16 ? kBS : p.block_size;
#pragma unroll
        for (int j = 0; j < kAppend; ++j) {
            const int64_t slot = app_slot[j];
            if ((uint64_t)slot >= (uint64_t)(p.num_blocks * bs)) continue;     // outside the pool: skipped
            const int64_t blk = BS16 ? slot / kBS : slot >> p.block_shift;
            const int64_t dst = (blk * p.sb + (slot - blk * bs) * p.ss) * (int64_t)sizeof(T) +
                                (i0 + j * 256 + (int)threadIdx.x) % CPR * 16;
            store16(const_cast<char*>(kbase) + dst, app_k[j]);
            store16(const_cast<char*>(vbase) + dst, app_v[j]);
        }
    };
    dma_tile(t_begin, ids, s_k0, s_v0);
    ids = tile_ids(t_begin + 1);
    // One tile: wait for this wave's DMA of tile kt, meet the other waves (their DMAs
    // have landed and they are done with tile kt-1, so its buffer is free), compute S^T,
    // start the DMA of tile kt+1 into the free buffer, then the softmax and P·V.
    auto tile = [&](int kt, const uint16_t* tile_k, const uint16_t* tile_v, uint16_t* nk, uint16_t* nv) {
        __builtin_amdgcn_s_waitcnt(0);
        lds_barrier();
        // None of this wave's rows sees the tile: it only stages.
        const bool sees = kt * kKT < wave_kmax;

        // ---- S^T for 64 keys: two 32-key MFMA tiles.
        // Both 32-key halves' K fragments first, then the two accumulators' MFMAs
        // interleaved, so each LDS read feeds MFMAs of both halves; the phase runs at
        // raised wave priority so the SIMD's other wave fills the gaps with its softmax
        // rather than holding these MFMAs back (config 4 chunks: 348.5 -> 341 us).
        __builtin_amdgcn_s_setprio(1);
        f32x16 st[2];
        if (sees) {
            u32x4 kf[2][DSTEPS];
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const char* kt0 = reinterpret_cast<const char*>(tile_k) + half * 32 * ROWB;
#pragma unroll
                for (int s = 0; s < DSTEPS; ++s) {
                    const uint4 a = *reinterpret_cast<const uint4*>(kt0 + koff[s]);
                    kf[half][s] = u32x4{a.x, a.y, a.z, a.w};
                }
            }
            st[0] = f32x16{};
            st[1] = f32x16{};
#pragma unroll
            for (int s = 0; s < DSTEPS; ++s) {
                st[0] = Mfma<T>::run(kf[0][s], qfrag[s], st[0]);
                st[1] = Mfma<T>::run(kf[1][s], qfrag[s], st[1]);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        // The next tile's DMA goes out after the S^T MFMAs (issued at the tile's top, it
        // delayed them: config 4 chunks 332 -> 325 us for the move, with the DMA still
        // visible to the compiler; 318 vs 310 us between the two places with it hidden).
        if (kt + 1 < t_end) {
            dma_tile(kt + 1, ids, nk, nv);
            ids = tile_ids(kt + 2);
        }
        if (!sees) return;
        // ---- causal mask only on tiles that cross the workgroup's first query position.
        if (kt * kKT + kKT - 1 > first_pos) {
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = kt * kKT + half * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                    if (key > my_pos) st[half][r] = kNegInf;
                }
        }
        // ---- tile max of this query over our 32 keys and the partner lane's 32.
        float mt = kNegInf;
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int r = 0; r < 16; ++r) mt = fmaxf(mt, st[half][r]);
        mt = max_across32(mt) * p.scale_log2;   // scale > 0: max commutes with it
        asm("" : "+v"(mt));   // mt stays rounded: m_run - mt below is not contracted into an fma
        // Raise the running max only when this tile exceeds it by more than 2^8.
        const bool raise = mt > m_run + kRescaleThreshold;
        const float m_new = raise ? mt : m_run;
        const float alpha = raise ? fast_exp2(m_run - mt) : 1.f;   // exp2(-inf) = 0 for m_run = -inf
        if (__builtin_amdgcn_ballot_w64(raise)) {
#pragma unroll
            for (int t = 0; t < DTILES; ++t) o[t] *= alpha;
        }
        m_run = m_new;
        // A query with no visible key yet keeps m = -inf; its scores are all -inf, so any
        // finite offset gives exp2(-inf) = 0 without a per-element select.
        const float m_off = m_new == kNegInf ? 0.f : m_new;
        float psum = 0.f;
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float e = fast_exp2(fmaf(st[half][r], p.scale_log2, -m_off));
                st[half][r] = e;
                psum += e;
            }
        psum = sum_across32(psum);
        l_run = l_run * alpha + psum;

        // ---- O^T += V^T · P^T, 16 keys per MFMA step. Step s uses accumulator
        // registers 8*(s%2) .. +8 of tile s/2: keys 16*(s%2) + 4h + {0..3} and +8.
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const f32x16& sv = st[s >> 1];
            const int r0 = 8 * (s & 1);
            const u32x4 pb = {Mfma<T>::pack(sv[r0 + 0], sv[r0 + 1]), Mfma<T>::pack(sv[r0 + 2], sv[r0 + 3]),
                              Mfma<T>::pack(sv[r0 + 4], sv[r0 + 5]), Mfma<T>::pack(sv[r0 + 6], sv[r0 + 7])};
            // This lane's 4-key groups: rows 4 (grp / 2) .. +3 and +8 .. +11 of the step's
            // 16-key group (lane groups 0-1: h = 0, groups 2-3: h = 1), in voff_lo / voff_hi.
            const char* vgrp = reinterpret_cast<const char*>(tile_v) + ((s >> 1) * 32 + 16 * (s & 1)) * ROWB;
#pragma unroll
            for (int t = 0; t < DTILES; ++t) {
                const uint2 lo = lds_read_tr16(reinterpret_cast<const uint16_t*>(vgrp + voff_lo[t]));
                const uint2 hi = lds_read_tr16(reinterpret_cast<const uint16_t*>(vgrp + voff_hi[t]));
                o[t] = Mfma<T>::run(u32x4{lo.x, lo.y, hi.x, hi.y}, pb, o[t]);
            }
        }
    };
    // Two tiles per trip, so every buffer reference names a fixed array.
    for (int kt = t_begin; kt < t_end; kt += 2) {
        tile(kt, s_k0, s_v0, s_k1, s_v1);
        if (kt + 1 < t_end) tile(kt + 1, s_k1, s_v1, s_k0, s_v0);
    }

    for (int i0 = 0; i0 < n_pieces; i0 += kAppend * 256) {
        append_load(i0);
        append_store(i0);
    }
    // ---- store: the lane holds d = 32 t + 8 (r/4) + 4 h + r%4 of its query row.
    if (!my_live) return;
    const int64_t tok = q_first + my_q;
    if (run < n_tiles) {
        // One of several splits: this row's partial, unnormalised.
        const int64_t row = tok * p.num_heads + my_head;
        const int64_t slot = row * p.splits + split;
        float* po = p.ws_o + slot * D + 4 * h;
#pragma unroll
        for (int t = 0; t < DTILES; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (32 * t + 8 * i < D)
                    *reinterpret_cast<float4*>(po + 32 * t + 8 * i) =
                        make_float4(o[t][4 * i], o[t][4 * i + 1], o[t][4 * i + 2], o[t][4 * i + 3]);
        if (h == 0) *reinterpret_cast<float2*>(p.ws_ml + slot * 2) = make_float2(m_run, l_run);
        // Splits that hold a key this row sees (the merge reads only those).
        if (p.ws_rows && h == 0 && split == 0) p.ws_rows[row] = my_pos / (run * kKT) + 1;
        return;
    }
    if (p.ws_rows && h == 0) p.ws_rows[tok * p.num_heads + my_head] = 0;   // finished here
    const float inv = 1.f / l_run;
    T* orow = reinterpret_cast<T*>(p.out) + tok * p.out_st + (int64_t)my_head * p.out_sh;
#pragma unroll
    for (int t = 0; t < DTILES; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (32 * t + 8 * i >= D) continue;
            const int d = 32 * t + 8 * i + 4 * h;
            const uint32_t w0 = Mfma<T>::pack(o[t][4 * i] * inv, o[t][4 * i + 1] * inv);
            const uint32_t w1 = Mfma<T>::pack(o[t][4 * i + 2] * inv, o[t][4 * i + 3] * inv);
            *reinterpret_cast<uint2*>(orow + d) = make_uint2(w0, w1);
        }
}

// Merge of the splits, launched after the kernel above on the same stream: D / 4 lanes per
// query row (four head_dim elements each), log-sum-exp rule over the row's splits in key
// order. Rows that one workgroup finished are marked 0 and skipped, as are tokens of no
// sequence (rows the launch above never wrote: tokens past query_start_loc's end). Bound by
// the latency of its two dependent loads and by workgroup launches, hence as many rows per
// wave as fit.
template <int D>
constexpr int kMergeRows = 4 * (64 / (D / 4));   // query rows per 256-thread workgroup

template <typename T, int D>
__global__ __launch_bounds__(256) void prefill_merge_kernel(const AttnParams p) {
    constexpr int LPR = D / 4, RPW = 64 / LPR;
    const int lane = lane_id();
    if (lane >= RPW * LPR) return;
    const int64_t row = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * RPW + lane / LPR;
    const int64_t end = p.qsl ? p.qsl[p.num_seqs] : p.num_tokens;
    if (row >= end * p.num_heads) return;
    const int64_t tok = row / p.num_heads;
    int n;
    if (p.qsl) {
        n = p.ws_rows[row];
    } else {
        // A decode batch: the splits of the row's own context, none if it has only one.
        const int64_t cap = p.table_width * p.block_size;
        int64_t c = p.ctx_lens[tok];
        c = c < cap ? c : cap;
        const int tiles = (int)((c + kKT - 1) / kKT);
        const int run = split_run(tiles, p.splits, p.split_tiles);
        n = run > 0 && run < tiles ? (tiles + run - 1) / run : 0;
    }
    if (n <= 0 || n > p.splits) return;
    const int d = 4 * (lane % LPR);
    const float2* ml = reinterpret_cast<const float2*>(p.ws_ml) + row * p.splits;
    const float* o = p.ws_o + row * p.splits * D + d;
    constexpr int CH = 8;   // splits whose loads are in flight together
    float M = kNegInf, L = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s0 = 0; s0 < n; s0 += CH) {
        float2 mlv[CH];
        float4 ov[CH];
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const bool in = s0 + j < n;
            mlv[j] = in ? ml[s0 + j] : make_float2(kNegInf, 0.f);
            ov[j] = in ? *reinterpret_cast<const float4*>(o + (int64_t)(s0 + j) * D) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        float Mc = M;
#pragma unroll
        for (int j = 0; j < CH; ++j) Mc = fmaxf(Mc, mlv[j].x);
        const float rescale = M == kNegInf ? 0.f : fast_exp2(M - Mc);
        L *= rescale;
        acc.x *= rescale;
        acc.y *= rescale;
        acc.z *= rescale;
        acc.w *= rescale;
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const float sc = mlv[j].x == kNegInf ? 0.f : fast_exp2(mlv[j].x - Mc);
            L += sc * mlv[j].y;
            acc.x += sc * ov[j].x;
            acc.y += sc * ov[j].y;
            acc.z += sc * ov[j].z;
            acc.w += sc * ov[j].w;
        }
        M = Mc;
    }
    T* orow = reinterpret_cast<T*>(p.out) + tok * p.out_st + (row - tok * p.num_heads) * p.out_sh + d;
    const float inv = 1.f / L;
    *reinterpret_cast<uint2*>(orow) =
        make_uint2(Mfma<T>::pack(acc.x * inv, acc.y * inv), Mfma<T>::pack(acc.z * inv, acc.w * inv));
}

// Workgroups of the flat grid, a multiple of 8: the splits' items, or room for every row
// tile the batch can hold (a sequence's last tile may be partial), whichever is more.
int64_t prefill_workgroups(const AttnParams& p) {
    const int64_t grid = ceil_div((int64_t)p.max_query_len * p.group, kRows) * p.num_seqs;
    const int64_t fill = p.num_tokens * p.group / kRows + p.num_seqs;
    int64_t items = (grid < fill || p.num_seqs > kPrefillSortSeqs ? grid : fill) * p.num_kv_heads;
    if (p.splits > 1 && p.split_items > items) items = p.split_items;
    return ceil_div(items, 8) * 8;
}

template <typename T, int D, bool BS16>
int launch_one(const AttnParams& p, hipStream_t stream) {
    const int64_t wgs = prefill_workgroups(p);
    if (wgs == 0) return PKV_OK;
    paged_prefill_kernel<T, D, BS16><<<dim3((unsigned)wgs), 256, 0, stream>>>(p);
    const int rc = check_launch("paged prefill attention");
    if (rc || p.splits == 1) return rc;
    const int64_t rows = p.num_tokens * p.num_heads;
    prefill_merge_kernel<T, D><<<dim3((unsigned)ceil_div(rows, kMergeRows<D>)), 256, 0, stream>>>(p);
    return check_launch("paged prefill merge");
}

template <typename T>
int launch_t(const AttnParams& p, hipStream_t stream) {
    const bool bs16 = p.block_size == kBS;
    switch (p.head_dim) {
        case 32: return launch_one<T, 32, false>(p, stream);
        case 48: return launch_one<T, 48, false>(p, stream);
        case 64: return bs16 ? launch_one<T, 64, true>(p, stream) : launch_one<T, 64, false>(p, stream);
        case 80: return launch_one<T, 80, false>(p, stream);
        case 96: return launch_one<T, 96, false>(p, stream);
        case 112: return launch_one<T, 112, false>(p, stream);
        case 128: return bs16 ? launch_one<T, 128, true>(p, stream) : launch_one<T, 128, false>(p, stream);
    }
    return PKV_EUNSUPPORTED;
}

}  // namespace

// The cheapest of a few run lengths in a model of the launch, in us, from per-workgroup
// time stamps: a workgroup takes kStart before and after its tiles and then a tile's time,
// 1.1 us alone and 1.9 us where the GPU is full (two workgroups per CU at head_dim 112 and
// 128, three at 80 and 96, four below: registers and LDS); once there are more workgroups
// than slots the last ones start late, half a workgroup's time on average; a split launch
// adds the merge kernel, and its partials' way to memory at ~4.5 TB/s.
SplitPlan prefill_split_plan(int64_t num_seqs, int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                             int64_t num_tokens, const int64_t* ctx, const int64_t* qlen, int64_t max_context_len) {
    constexpr float kStart = 6.f, kTileAlone = 1.1f, kTileFull = 1.9f, kMerge = 4.f, kBytesPerUs = 4.5e6f;
    constexpr float kWorth = 0.85f;              // the gain that a split has to promise
    constexpr int64_t kMaxBytes = 128 << 20;     // of workspace, the counters' room and roundings included
    static const int kRuns[] = {4, 5, 6, 8, 10, 12, 14, 17, 20, 24, 28, 34, 40, 48, 56, 68, 80, 96, 112, 136, 160, 192};
    SplitPlan plan{1, 0x7fffffff, 0, 0, 0, 0};
    if (num_seqs < 1 || num_seqs > kPrefillSortSeqs || num_tokens < 1 || num_kv_heads < 1 || head_dim < 1) return plan;
    const int64_t group = num_heads / num_kv_heads;
    const int64_t slots = head_dim >= 112 ? 512 : head_dim >= 80 ? 768 : 1024;
    auto launch_us = [&](int64_t wgs, int64_t longest, int64_t work) {
        const float full = wgs < slots ? (float)wgs / slots : 1.f;
        const float tile = kTileAlone + (kTileFull - kTileAlone) * full;
        const float one = longest * tile + kStart;
        if (wgs <= slots) return one;
        const float all = (work * tile + wgs * kStart) / slots + 0.5f * one;
        return all > one ? all : one;
    };
    // Per sequence with work: key tiles, workgroups unsplit, query rows of all KV heads.
    static_assert(kPrefillSortSeqs % 4 == 0, "");
    double tiles[kPrefillSortSeqs], per_split[kPrefillSortSeqs], rows_of[kPrefillSortSeqs];
    int live = 0;
    int64_t wgs = 0, work = 0, longest = ctx ? 0 : (max_context_len + kKT - 1) / kKT;
    for (int64_t i = 0; i < num_seqs; ++i) {
        // Without the lengths (a decode call): contexts spread evenly up to the bound.
        const int64_t c = ctx ? ctx[i] : max_context_len * (2 * i + 1) / (2 * num_seqs);
        const int64_t r = (qlen ? qlen[i] : 1) * group;
        if (c <= 0 || r <= 0) continue;
        const int64_t t = c < ((int64_t)1 << 36) ? (c + kKT - 1) / kKT : (int64_t)1 << 30;
        const int64_t w = (r + kRows - 1) / kRows * num_kv_heads;
        wgs += w;
        work += w * t;
        longest = longest > t ? longest : t;
        if (wgs >= 2 * slots) return plan;       // the GPU is full, and stays so
        tiles[live] = (double)t;
        per_split[live] = (double)w;
        rows_of[live++] = (double)(r * num_kv_heads);
    }
    if (longest * kKT <= kSplitMinContext) return plan;
    for (int i = live; i % 4; ++i) {             // nothing, for the loop below
        tiles[i] = 1.0;
        per_split[i] = rows_of[i] = 0.0;
    }
    const int64_t rows = num_tokens * num_heads;
    float best = kWorth * launch_us(wgs, longest, work);
    for (const int64_t run : kRuns) {
        if (run >= longest) break;
        const int64_t splits = ceil_div(longest, run);
        if (kMergeCounterBytes + 3 * 256 + rows * 4 + rows * splits * (head_dim + 2) * 4 > kMaxBytes) continue;
        // The least that it can take, from the sums alone: mostly enough to pass on.
        const int64_t least = ceil_div(work, run) > wgs ? ceil_div(work, run) : wgs;
        if (launch_us(least, ceil_div(longest, splits), work) + kMerge >= best) continue;
        // In doubles and four sums, for the host's vector units (22 run lengths over 256
        // sequences: 30-50 us in 64-bit integers); all are whole numbers below 2^53.
        const double inv = 1.0 / (double)run, above = (double)run - 0.5;
        auto splits_of = [&](double t) { return (double)(int32_t)((t + above) * inv); };
        double ns[4] = {}, ps[4] = {};
        for (int i = 0; i < live; i += 4)
            for (int j = 0; j < 4; ++j) {
                // ceil(tiles / run): the half keeps the product off whole numbers.
                const double s = splits_of(tiles[i + j]);
                ns[j] += per_split[i + j] * s;
                ps[j] += s > 1 ? rows_of[i + j] * s : 0.0;
            }
        const double n = ns[0] + ns[1] + ns[2] + ns[3], parts = ps[0] + ps[1] + ps[2] + ps[3];
        // The longest of the even splits, rounded up; no split is longer than the run.
        double top = 0;
        for (int i = 0; i < live && top <= (double)run - 1.0; ++i)
            if (tiles[i] > top) {
                const double even = tiles[i] / splits_of(tiles[i]);
                top = even > top ? even : top;
            }
        top += 1.0 - 1e-9;
        const float us = launch_us((int64_t)n, (int64_t)top, work) + kMerge +
                         (int64_t)parts * (head_dim + 2) * 4 / kBytesPerUs;
        if (us >= best) continue;
        best = us;
        plan.splits = (int)splits;
        plan.split_tiles = (int)run;
        plan.items = ctx ? (int64_t)n : wgs * splits;     // lengths unknown: room for all of them at the bound
    }
    if (plan.splits == 1) return plan;
    auto round256 = [](int64_t b) { return ceil_div(b, 256) * 256; };
    plan.rows_bytes = round256(rows * 4);
    plan.ml_bytes = round256(rows * plan.splits * 8);
    plan.o_bytes = round256(rows * plan.splits * head_dim * 4);
    return plan;
}

bool prefill_shape(int64_t block_size, int64_t head_dim, int dtype) {
    if (block_size < 8 || (block_size & (block_size - 1))) return false;
    if (head_dim % 16 || head_dim < 32 || head_dim > 128) return false;
    return dtype == PKV_FLOAT16 || dtype == PKV_BFLOAT16;
}

bool prefill_tuned(const AttnParams& p, int dtype) {
    if (!prefill_shape(p.block_size, p.head_dim, dtype)) return false;
    // The kernel's offsets are unsigned (strides too large for 32 bits take its per-row path).
    if (p.ss < 0) return false;
    // The kernel masks to -inf and takes the maximum before it scales: scale > 0 only.
    if (!(p.scale > 0.f)) return false;
    // The grid is one dimension, and row numbers of a sequence stay below 2^31.
    if (prefill_workgroups(p) > 0x7fffffff) return false;
    if (((int64_t)p.max_query_len + kRows) * p.group > 0x7fffffff) return false;
    // Masked-off rows are staged from a valid row of the pool: needs a non-empty pool.
    if (p.num_blocks < 1) return false;
    // 16-byte rows and 8-byte output stores need aligned pointers and strides; so do the
    // source rows of a fused append, which are staged by the same 16-byte DMA.
    uint64_t probe = (uint64_t)(uintptr_t)p.q | (uint64_t)(uintptr_t)p.k | (uint64_t)(uintptr_t)p.v |
                     (uint64_t)(uintptr_t)p.out | (uint64_t)(p.q_st * 2) | (uint64_t)(p.q_sh * 2) |
                     (uint64_t)(p.sb * 2) | (uint64_t)(p.ss * 2) | (uint64_t)(p.sh * 2) |
                     (uint64_t)(p.out_st * 2) | (uint64_t)(p.out_sh * 2);
    if (p.app_k)
        probe |= (uint64_t)(uintptr_t)p.app_k | (uint64_t)(uintptr_t)p.app_v | (uint64_t)(p.app_st * 2) |
                 (uint64_t)(p.app_sh * 2);
    return probe % 16 == 0;
}

int launch_prefill_attention(const AttnParams& p, int dtype, hipStream_t stream) {
    if (!prefill_tuned(p, dtype)) return PKV_EUNSUPPORTED;
    if (p.num_seqs == 0 || p.num_tokens == 0) return PKV_OK;
    if (dtype == PKV_FLOAT16) return launch_t<_Float16>(p, stream);
    return launch_t<bf16_t>(p, stream);
}

}  // namespace pkv
