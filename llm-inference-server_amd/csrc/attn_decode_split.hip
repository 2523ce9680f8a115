// Paged decode attention on MFMA (gfx950) in one launch, fp32/fp16/bf16, head_dim a multiple
// of 16 from 32 to 128, GQA groups up to 16, block sizes that are powers of two from 8 up.
// Takes every such decode batch, in 16 bits below the size from which the persistent kernel
// (attn_decode_mfma.hip) is the better one.
//
// Bound: HBM for batches of tens of MB, latency below that. Every K/V byte is read once
// (all heads of a group share the read); what the launch pays on top is its start (lengths,
// block ids, the first K/V rows: three dependent memory round trips), the tail of unequal
// contexts, and the merge of split contexts. Hence:
//
//  * Work unit: one workgroup = (sequence, KV head, run of 16-key units) x NW waves; wave w
//    takes units w, w + NW, ... of the run. A batch of few (sequence, KV head) pairs gets
//    workgroups of more waves (the launch picks NW), so short contexts need no split.
//  * Runs are cut on the device: every wave sums the batch's units, takes the shortest run
//    length (no less than 4 units a wave) with which all runs fit the GPU at once, and finds
//    its own (sequence, split) by a wave scan, no barrier. The grid is bounded by the GPU, not
//    by the longest context a captured graph must serve, and holds next to no empty
//    workgroups; a sequence's runs are of even lengths. Batches that fill the GPU by their
//    pairs alone have only their outlying long contexts cut (pick_long).
//  * Streaming: per wave a two-slot ring of units in LDS (K and V, 16 rows of one KV head),
//    filled by nontemporal LDS DMA; a unit's K and V^T fragments are read into registers
//    first and the slot refilled with the unit after next at once. Waits are explicit vmcnt
//    counts; DMAs and ring reads are inline asm, unseen by the compiler's wait counting.
//  * Contraction (Contract), in 16 bits as in the persistent kernel: S^T = K Q^T on 16x16x32, P^T straight from the
//    accumulator into O^T += V^T P^T on 16x16x16, V^T by the transposing LDS read. 12 MFMAs
//    and ~80 VALU instructions per unit at head_dim 128, where v_dot2 arithmetic took ~900.
//    fp32 on 16x16x4.
//  * fp32 prompts of few query rows, or of shapes without another kernel, take the same
//    kernel with 16 (token, head) rows in place of one token's heads. us a call with the
//    append: 8 prompts of 1-150 tokens behind up to 1,000, 12/4 heads of 80, block size 32,
//    1,000 -> 44; 16 of 1-200 behind up to 1,500, 24/8 heads of 32, block size 8, 3,295 -> 73.
//  * Merge: the waves' partials meet in LDS; split contexts leave fp32 partials that the
//    last workgroup of each (sequence, KV head) to finish merges in run order (agent-scope
//    stores, one counter, no workgroup ever waits for another).
//  * Fused append: the new token's row is staged from the caller's rows by the DMA of the
//    context's last unit, and goes to its pool slot from registers, so nothing waits for the
//    store.
//
// Numerics follow the reference gather path (core/attention.py:130-153) as the persistent
// kernel does: scores rounded to the pool dtype before and after the scale, softmax in fp32,
// probabilities exp2(s - m) rounded to the pool dtype before P·V, fp32 accumulation, one
// rounding of the output. Keys at or beyond context_lens are never loaded.
// m is the maximum of the unit itself in 16 bits: its largest weight is then 1, which rounds to
// itself, and the unit's product is scaled to the running maximum (raised lazily, past 2^8
// only) in fp32. Against 64 bits, before that (weights against the running maximum) and now:
// 12 layers of a GPT-2 step 4.30e-4 -> 4.16e-4, 64 GPT-2 sequences 8.45e-4 -> 8.34e-4, 24/8
// heads of 128 in blocks of 32 1.439e-3 -> 1.432e-3; it costs 0-0.3 us a call (8 GPT-2
// sequences of 16-1000 tokens 8.3 -> 8.7 us).
#include "attention.h"

namespace pkv {
namespace {

constexpr int kUnit = 16;                     // keys per unit
constexpr float kLazyMax = 8.f;               // base 2
constexpr int kMaxScanSeqs = 1024;            // sequences a wave scans (16 per lane)
constexpr int kScanPer = kMaxScanSeqs / 64;
constexpr int kCus = 256;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// 16-byte LDS read / transposing LDS read (ds_read_b64_tr_b16: within 16 lanes, source lane c
// pointing at V[key0 + c / 4][d0 + 4 (c % 4)], lane i receives V[key0 .. key0 + 3][d0 + i]).
__device__ __forceinline__ u32x4 lds_read16(const char* ptr) {
    const uint4 v = *reinterpret_cast<const uint4*>(ptr);
    return u32x4{v.x, v.y, v.z, v.w};
}
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint2 lds_read_tr16(const char* ptr) {
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(ptr));
    return __builtin_bit_cast(uint2, v);
}
// Waits that also keep the compiler's memory operations on their side: the ring's DMAs are
// unseen by it, so nothing else orders LDS reads against them.
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// The contraction of one unit, from its ring slot. MFMA lane layouts as pinned for the
// persistent kernel (attn_decode_mfma.hip): 16x16xK puts A[i][k] in lane i + 16 (k / (K/4)),
// B[k][j] in lane j + 16 (k / (K/4)), D[i][j] in lane j + 16 (i / 4), register i % 4.
template <typename T>
struct Half {
    __device__ __forceinline__ static uint32_t pack(float lo, float hi);
    __device__ __forceinline__ static f32x4 qk(u32x4 a, u32x4 b, f32x4 c);
    __device__ __forceinline__ static f32x4 pv(uint2 a, uint2 b, f32x4 c);
    __device__ __forceinline__ static float round(float x);
};
template <>
struct Half<bf16_t> {
    __device__ __forceinline__ static f32x4 qk(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                       c, 0, 0, 0);
    }
    __device__ __forceinline__ static f32x4 pv(uint2 a, uint2 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(bf16x4, a), __builtin_bit_cast(bf16x4, b),
                                                         c, 0, 0, 0);
    }
    __device__ __forceinline__ static uint32_t pack(float lo, float hi) {
        bf16x2_t v = {(__bf16)lo, (__bf16)hi};
        return __builtin_bit_cast(uint32_t, v);
    }
    __device__ __forceinline__ static float round(float x) { return (float)(__bf16)x; }
};
template <>
struct Half<_Float16> {
    __device__ __forceinline__ static f32x4 qk(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                      0, 0, 0);
    }
    __device__ __forceinline__ static f32x4 pv(uint2 a, uint2 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c,
                                                     0, 0, 0);
    }
    __device__ __forceinline__ static uint32_t pack(float lo, float hi) {
        half2_t v = {(_Float16)lo, (_Float16)hi};
        return __builtin_bit_cast(uint32_t, v);
    }
    __device__ __forceinline__ static float round(float x) { return (float)(_Float16)x; }
};

// 16-bit pools: S^T on 16x16x32 (the K read of step j gives a lane 8 dims), O^T on 16x16x16
// from the transposing V read, probabilities in the pool dtype.
template <typename T, int D>
struct Contract {
    static constexpr int KS = (D + 31) / 32;  // 16-byte K (and Q) pieces per lane
    static constexpr int VT = D / 16;
    static constexpr int CPR = D * 2 / 16;
    // Physical 16-byte slot of logical chunk c of ring row r is c ^ swizzle(r): the 16 rows
    // of a K read fall in different banks (at head_dim 48, 80 and 112 in pairs).
    __device__ __forceinline__ static int swizzle(int r) {
        if constexpr (D == 128) return ((r & 3) << 2) | ((r >> 2) & 3);
        else if constexpr (D == 64) return (((r >> 1) & 1) << 2) | (((r >> 2) & 1) << 1) | ((r >> 3) & 1);
        else if constexpr (D % 32 == 0) return (r >> 2) & 3;
        else return (r >> 3) & 1;
    }
    __device__ __forceinline__ static int k_chunk(int j, int lg) { return 4 * j + lg; }
    u32x4 kf[KS];
    uint2 vf[VT];
    uint32_t k_addr[KS], v_addr[VT];
    // Per-lane addresses inside a unit: K row ln, chunk 4 j + lg (one past head_dim re-reads
    // another and is zeroed); V^T rows 4 lg + ln / 4, columns 16 t + 4 (ln % 4).
    __device__ __forceinline__ void address(int lg, int ln) {
#pragma unroll
        for (int j = 0; j < KS; ++j) {
            const int c = 4 * j + lg < CPR ? 4 * j + lg : 4 * j + (lg & 1);
            k_addr[j] = (uint32_t)(ln * D * 2 + ((c ^ swizzle(ln)) << 4));
        }
        const int row = 4 * lg + (ln >> 2);
#pragma unroll
        for (int t = 0; t < VT; ++t)
            v_addr[t] = (uint32_t)(row * D * 2 + (((2 * t + ((ln & 3) >> 1)) ^ swizzle(row)) << 4) + 8 * (ln & 1));
    }
    __device__ __forceinline__ void read(const char* k, const char* v, int lg) {
#pragma unroll
        for (int j = 0; j < KS; ++j) kf[j] = lds_read16(k + k_addr[j]);
#pragma unroll
        for (int t = 0; t < VT; ++t) vf[t] = lds_read_tr16(v + v_addr[t]);
        wait_lds();
        if constexpr (D % 32 != 0)
            if (lg >= 2) kf[KS - 1] = u32x4{0u, 0u, 0u, 0u};
    }
    __device__ __forceinline__ f32x4 scores(const u32x4 (&qf)[KS]) const {
        f32x4 st = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < KS; ++j) st = Half<T>::qk(kf[j], qf[j], st);
        return st;
    }
    __device__ __forceinline__ static float scaled(float dot, float scale) {
        return Half<T>::round(Half<T>::round(dot) * scale) * kLog2e;
    }
    __device__ __forceinline__ void accumulate(const float (&pr)[4], float sc, f32x4 (&o)[VT]) const {
        const uint2 pb = make_uint2(Half<T>::pack(pr[0], pr[1]), Half<T>::pack(pr[2], pr[3]));
#pragma unroll
        for (int t = 0; t < VT; ++t) o[t] += Half<T>::pv(vf[t], pb, f32x4{0.f, 0.f, 0.f, 0.f}) * sc;
    }
    __device__ __forceinline__ static void store4(T* to, float4 v, bool wide) {
        const uint32_t w0 = Half<T>::pack(v.x, v.y), w1 = Half<T>::pack(v.z, v.w);
        if (wide) {
            *reinterpret_cast<uint2*>(to) = make_uint2(w0, w1);
        } else {
            uint16_t* o16 = reinterpret_cast<uint16_t*>(to);
            o16[0] = (uint16_t)w0;
            o16[1] = (uint16_t)(w0 >> 16);
            o16[2] = (uint16_t)w1;
            o16[3] = (uint16_t)(w1 >> 16);
        }
    }
};

// fp32 pools: 16x16x4, one element per lane and step. S^T: a 16-byte K read gives a lane four
// dims, one for each of four steps (Q^T is held in the same order). O^T: step r takes keys
// 4 lg + r, whose probabilities are accumulator register r as it stands; V^T by 4-byte reads.
// Nothing is rounded below fp32.
template <int D>
struct Contract<float, D> {
    static constexpr int KS = D / 16;
    static constexpr int VT = D / 16;
    static constexpr int CPR = D * 4 / 16;
    // Conflict-free at D = 64 and 128: the 16 rows of a K read go to 16 slots, the rows 4 lg + r
    // of a V read to four different 64-byte groups.
    __device__ __forceinline__ static int swizzle(int r) {
        if constexpr (D % 64 == 0) return r & 15;
        else if constexpr (D == 32) return r & 7;
        else return r & 3;
    }
    __device__ __forceinline__ static int k_chunk(int j, int lg) { return 4 * j + lg; }
    u32x4 kf[KS];
    float vf[4][VT];
    uint32_t k_addr[KS];
    int lg_, ln_;
    __device__ __forceinline__ void address(int lg, int ln) {
#pragma unroll
        for (int j = 0; j < KS; ++j) k_addr[j] = (uint32_t)(ln * D * 4 + (((4 * j + lg) ^ swizzle(ln)) << 4));
        lg_ = lg;
        ln_ = ln;
    }
    __device__ __forceinline__ void read(const char* k, const char* v, int) {
#pragma unroll
        for (int j = 0; j < KS; ++j) kf[j] = lds_read16(k + k_addr[j]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 4 * lg_ + r;
#pragma unroll
            for (int t = 0; t < VT; ++t)
                vf[r][t] = *reinterpret_cast<const float*>(v + row * D * 4 + (((4 * t + (ln_ >> 2)) ^ swizzle(row)) << 4) +
                                                           4 * (ln_ & 3));
        }
        wait_lds();
    }
    __device__ __forceinline__ f32x4 scores(const u32x4 (&qf)[KS]) const {
        // Eight chains, summed as a tree: shorter ones are faster (each step waits for the one
        // before it) and lose less (a score's rounding errors are the output's).
        f32x4 st[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) st[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < KS; ++j) {
            const f32x4 a = __builtin_bit_cast(f32x4, kf[j]), b = __builtin_bit_cast(f32x4, qf[j]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                st[4 * (j & 1) + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], st[4 * (j & 1) + e], 0, 0, 0);
        }
        return ((st[0] + st[1]) + (st[2] + st[3])) + ((st[4] + st[5]) + (st[6] + st[7]));
    }
    __device__ __forceinline__ static float scaled(float dot, float scale) { return ref_score_log2<float>(dot, scale); }
    __device__ __forceinline__ void accumulate(const float (&pr)[4], float, f32x4 (&o)[VT]) const {
#pragma unroll
        for (int t = 0; t < VT; ++t) {
            f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int r = 0; r < 4; ++r) a = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[r][t], pr[r], a, 0, 0, 0);
            o[t] += a;
        }
    }
    __device__ __forceinline__ static void store4(float* to, float4 v, bool wide) {
        if (wide) {
            *reinterpret_cast<float4*>(to) = v;
        } else {
            to[0] = v.x;
            to[1] = v.y;
            to[2] = v.z;
            to[3] = v.w;
        }
    }
};

__device__ __forceinline__ uint32_t lds_addr(const void* ptr) {
    return (uint32_t)(uintptr_t)((const __attribute__((address_space(3))) char*)ptr);
}

// 16 bytes per lane HBM -> LDS address lds + 16 lane, nontemporal (read once: a stream of
// this pattern runs 12% faster so). M0 belongs to these helpers alone in this kernel.
__device__ __forceinline__ void dma16_nt(const char* sbase, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                 :
                 : "s"(lds), "v"(voff), "s"(sbase)
                 : "memory");
}
__device__ __forceinline__ void dma16_nt(const char* addr, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt"
                 :
                 : "s"(lds), "v"(addr)
                 : "memory");
}

// ------------------------------------------------------------------ wave scans (int)
template <int CTRL>
__device__ __forceinline__ int dpp_shr(int x) {   // 0 where the source is outside the row
    return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, true);
}
// Inclusive sum over lanes 0 .. l, in every lane l.
__device__ __forceinline__ int wave_scan(int x, int lane) {
    x += dpp_shr<0x111>(x);   // row_shr:1, 2, 4, 8 within rows of 16
    x += dpp_shr<0x112>(x);
    x += dpp_shr<0x114>(x);
    x += dpp_shr<0x118>(x);
    const int r0 = __builtin_amdgcn_readlane(x, 15), r1 = __builtin_amdgcn_readlane(x, 31),
              r2 = __builtin_amdgcn_readlane(x, 47);
    return x + (lane >= 16 ? r0 : 0) + (lane >= 32 ? r1 : 0) + (lane >= 48 ? r2 : 0);
}
__device__ __forceinline__ int wave_total(int x, int lane) {
    return __builtin_amdgcn_readlane(wave_scan(x, lane), 63);
}
// The largest of the lanes' x >= 0.
__device__ __forceinline__ int wave_max(int x) {
    auto up = [](int a, int b) { return a > b ? a : b; };
    x = up(x, dpp_shr<0x111>(x));
    x = up(x, dpp_shr<0x112>(x));
    x = up(x, dpp_shr<0x114>(x));
    x = up(x, dpp_shr<0x118>(x));
    return up(up(__builtin_amdgcn_readlane(x, 15), __builtin_amdgcn_readlane(x, 31)),
              up(__builtin_amdgcn_readlane(x, 47), __builtin_amdgcn_readlane(x, 63)));
}

// Context length as every decode kernel clamps it: never past the table row or the
// partials the workspace was sized for (neither binds for valid input).
__device__ __forceinline__ int decode_ctx(const AttnParams& p, int seq) {
    const int64_t cap = p.table_width * (int64_t)p.block_size;
    const int64_t parts = (int64_t)p.max_parts * kDecodePart;
    int64_t c = p.ctx_lens[seq];
    c = c < cap ? c : cap;
    c = c < parts ? c : parts;
    return c > 0 ? (int)c : 0;
}

// How a launch cuts its contexts (lengths in units). The host gives what the shape decides; the
// lengths decide the rest on the device, so that a sequence's result does not depend on the
// bound that the launch was given for them: a captured step, told the longest context its
// tables allow, computes what the eager step computes.
enum CutMode { kCutNone, kCutRuns, kCutLong };
struct Cut {
    int mode;
    int min_run;                              // a run is never shorter
    int whole;                                // a batch of no longer context is not cut
    int slots, slots2, slots2_from;           // runs of one KV head that the GPU holds (0: do not
                                              // cut); slots2 where the longest context reaches slots2_from
    int long_from;                            // kCutLong: only contexts from here on are cut
};

// The `at`-th run of one KV head's batch, numbered sequence by sequence; seq < 0: none.
struct Pick {
    int seq, ctx, split, n_splits;
};

// Every wave by itself, lane l holding the contexts of sequences PER l .. PER l + PER - 1.
template <int PER>
__device__ __forceinline__ Pick pick_run(const AttnParams& p, int lane, int at, const Cut& cut) {
    int units_of[PER], cl[PER], units = 0, longest = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int s = lane * PER + i;
        cl[i] = s < p.num_seqs ? decode_ctx(p, s) : 0;
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        units_of[i] = (cl[i] + kUnit - 1) / kUnit;
        units += units_of[i];
        longest = units_of[i] > longest ? units_of[i] : longest;
    }
    // In whole partials, as the host rounds the bound.
    constexpr int PART = kDecodePart / kUnit;
    longest = (wave_max(longest) + PART - 1) / PART * PART;
    const int slots = longest <= cut.whole ? 0 : longest >= cut.slots2_from ? cut.slots2 : cut.slots;
    // The shortest run with which one KV head's runs fit its share of the GPU's slots: from
    // the even share of those left when every sequence's last run is half empty, up in
    // growing steps (mostly none or one).
    const int total = wave_total(units, lane);
    int run = 1 << 30;                        // none is cut
    if (slots > 0) {
        const int even = slots - p.num_seqs / 2;  // slots >= num_seqs
        run = (total + even - 1) / even;
        run = run > cut.min_run ? run : cut.min_run;
    }
    int n_of[PER], mine = 0;
    for (int step = (run + 15) >> 4;; run += step, step += (step + 1) >> 1) {
        mine = 0;
        const float inv = 1.f / (float)run;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            // ceil(units / run): exact after one correction either way.
            const int u = units_of[i];
            int q = (int)((float)u * inv);
            q -= q * run > u ? 1 : 0;
            q += (q + 1) * run <= u ? 1 : 0;
            n_of[i] = q + (q * run < u ? 1 : 0);
            mine += n_of[i];
        }
        if (run >= total || wave_total(mine, lane) <= slots) break;
    }
    const int incl = wave_scan(mine, lane);
    const uint64_t found = __builtin_amdgcn_ballot_w64(at < incl);
    if (!found) return Pick{-1, 0, 0, 0};
    const int src = __builtin_ctzll(found);   // the first lane whose runs reach past `at`
    int left = at - (__builtin_amdgcn_readlane(incl, src) - __builtin_amdgcn_readlane(mine, src));
    if constexpr (PER == 1) {
        return Pick{src, __builtin_amdgcn_readlane(cl[0], src), left, __builtin_amdgcn_readlane(n_of[0], src)};
    } else {
        Pick r{-1, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (r.seq < 0) {
                const int n = __builtin_amdgcn_readlane(n_of[i], src);
                if (left < n) r = Pick{src * PER + i, __builtin_amdgcn_readlane(cl[i], src), left, n};
                else left -= n;
            }
        return r;
    }
}

// Batches that fill the GPU by themselves (or exceed the scan above): only contexts that would
// outlast the rest of the launch are cut, into runs of twice a slot's share of the batch. The
// first num_seqs picks are the sequences' first runs, which read nothing but their own length
// unless it is a long one; the others are the further runs of the long ones, at most half as
// many as one KV head has slots. us a call before and now, 8/2 heads of 128, bf16, one context
// of 8192 tokens among 600 of 50-150: 92 -> 30, among 1100: 97 -> 41; fp32, one of 4096 among
// 400: 125 -> 61; 600 short ones alone 17.3 -> 17.1.
__device__ __forceinline__ Pick pick_long(const AttnParams& p, int lane, int at, const Cut& cut) {
    auto units_at = [&](int s) { return (decode_ctx(p, s) + kUnit - 1) / kUnit; };
    if (at < p.num_seqs) {
        const int ctx = __builtin_amdgcn_readfirstlane(decode_ctx(p, at));
        if (ctx == 0) return Pick{-1, 0, 0, 0};
        if ((ctx + kUnit - 1) / kUnit < cut.long_from) return Pick{at, ctx, 0, 1};
    }
    int sum = 0;
#pragma unroll 4
    for (int s = lane; s < p.num_seqs; s += 64) sum += units_at(s);
    const int share = (wave_total(sum, lane) + cut.slots - 1) / cut.slots;
    const int run = 2 * share > cut.min_run ? 2 * share : cut.min_run;
    auto runs_of = [&](int units) { return units >= cut.long_from ? (units + run - 1) / run : 1; };
    if (at < p.num_seqs) {
        const int ctx = __builtin_amdgcn_readfirstlane(decode_ctx(p, at));
        return Pick{at, ctx, 0, runs_of((ctx + kUnit - 1) / kUnit)};
    }
    int left = at - p.num_seqs;
    for (int s0 = 0; s0 < p.num_seqs; s0 += 64) {
        const int s = s0 + lane;
        const int ctx = s < p.num_seqs ? decode_ctx(p, s) : 0;
        const int more = runs_of((ctx + kUnit - 1) / kUnit) - 1;
        const int incl = wave_scan(more, lane);
        const uint64_t found = __builtin_amdgcn_ballot_w64(left < incl);
        if (found) {
            const int src = __builtin_ctzll(found);
            const int n = __builtin_amdgcn_readlane(more, src);
            return Pick{s0 + src, __builtin_amdgcn_readlane(ctx, src),
                        left - (__builtin_amdgcn_readlane(incl, src) - n) + 1, n + 1};
        }
        left -= __builtin_amdgcn_readlane(incl, 63);
    }
    return Pick{-1, 0, 0, 0};
}

// Prompts: the `at`-th tile of 16 query rows of one KV head's batch, numbered sequence by
// sequence; seq < 0: none. Same lanes as above.
struct PickTile {
    int seq, q_len, tile;
    int64_t q_first;
};
template <int PER>
__device__ __forceinline__ PickTile pick_tile(const AttnParams& p, int lane, int at) {
    int n_of[PER], ql[PER], mine = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int s = lane * PER + i;
        ql[i] = s < p.num_seqs ? (int)(p.qsl[s + 1] - p.qsl[s]) : 0;
        n_of[i] = ql[i] > 0 ? (int)(((uint32_t)ql[i] * (uint32_t)p.group + kUnit - 1) / kUnit) : 0;
        mine += n_of[i];
    }
    const int incl = wave_scan(mine, lane);
    const uint64_t found = __builtin_amdgcn_ballot_w64(at < incl);
    PickTile r{-1, 0, 0, 0};
    if (!found) return r;
    const int src = __builtin_ctzll(found);
    int left = at - (__builtin_amdgcn_readlane(incl, src) - __builtin_amdgcn_readlane(mine, src));
#pragma unroll
    for (int i = 0; i < PER; ++i)
        if (r.seq < 0) {
            const int n = __builtin_amdgcn_readlane(n_of[i], src);
            if (left < n) r = PickTile{src * PER + i, __builtin_amdgcn_readlane(ql[i], src), left, 0};
            else left -= n;
        }
    if (r.seq >= 0) r.q_first = p.qsl[r.seq];
    return r;
}

// LDS bytes of a workgroup (the ring; the merge's partials reuse it) and how many a CU holds.
constexpr int wgs_per_cu(int row_bytes, int NW) {
    const int ring = NW * 2 * 2 * kUnit * row_bytes;
    const int lds = (160 * 1024) / (ring + NW * 128 + 16), waves = 16 / NW;
    const int n = lds < waves ? lds : waves;
    return n < 1 ? 0 : n;
}

// PROMPT: the 16 rows are (token, head) pairs of a prompt, row f of a sequence being token
// f / G, head f % G, each with its own causal bound; no split and no append. Else they are
// the G heads of a sequence's one token.
template <typename T, int D, int NW, bool PROMPT>
__global__ __launch_bounds__(NW * 64) void paged_decode_split_kernel(const AttnParams p, const Cut cut) {
    using C = Contract<T, D>;
    constexpr int ISZ = (int)sizeof(T);
    constexpr int ROWB = D * ISZ;             // bytes per (token, head) row
    constexpr int CPR = ROWB / 16;            // 16-byte chunks per row
    constexpr int IPB = (kUnit * CPR + 63) / 64;   // DMA instructions per unit, K or V
    constexpr bool kWhole = kUnit * CPR % 64 == 0;
    constexpr bool kHalf = 64 % CPR == 0 && 64 / CPR <= 8;   // one 8-row half per instruction
    constexpr int KS = C::KS, VT = C::VT;
    constexpr int NT = NW * 64;
    constexpr int UB = kUnit * ROWB;          // bytes of a unit, K or V

    __shared__ __attribute__((aligned(1024))) char s_ring[NW][2][2][UB];   // [wave][slot][K, V]
    __shared__ float s_ml[NW][16][2];
    __shared__ uint32_t s_arrived;

    const int tid = (int)threadIdx.x;
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int KV = p.num_kv_heads, G = p.group;
    const int kvh = (int)(blockIdx.x % (uint32_t)KV);
    const int at = (int)(blockIdx.x / (uint32_t)KV);

    // ---- this workgroup's (sequence, run)
    int seq, ctx, split = 0, n_splits = 1;
    int rows = G, row0 = 0, pos0 = 0;         // query rows, the first one's number, token 0's position
    int64_t q_first = 0;
    if constexpr (PROMPT) {
        const PickTile pick = p.num_seqs <= 64 ? pick_tile<1>(p, lane, at) : pick_tile<kScanPer>(p, lane, at);
        if (pick.seq < 0) return;
        seq = pick.seq;
        q_first = pick.q_first;
        row0 = pick.tile * kUnit;
        rows = pick.q_len * G - row0 < kUnit ? pick.q_len * G - row0 : kUnit;
        pos0 = __builtin_amdgcn_readfirstlane(decode_ctx(p, seq)) - pick.q_len;
        // Keys visible to the tile's last token.
        ctx = pos0 + (int)((uint32_t)(row0 + rows - 1) / (uint32_t)G) + 1;
        if (ctx <= 0) return;
    } else if (cut.mode == kCutNone) {               // one workgroup per (sequence, KV head)
        seq = at;
        ctx = __builtin_amdgcn_readfirstlane(decode_ctx(p, seq));
        if (ctx == 0) return;
    } else {
        const Pick pick = cut.mode == kCutLong ? pick_long(p, lane, at, cut)
                          : p.num_seqs <= 64   ? pick_run<1>(p, lane, at, cut)
                                               : pick_run<kScanPer>(p, lane, at, cut);
        if (pick.seq < 0) return;
        seq = pick.seq;
        ctx = pick.ctx;
        split = pick.split;
        n_splits = pick.n_splits;
    }
    const int n_units = (ctx + kUnit - 1) / kUnit;
    const int run = (n_units + n_splits - 1) / n_splits;   // even runs
    n_splits = (n_units + run - 1) / run;
    if (split >= n_splits) return;            // an even cut took one run fewer
    const int u_end = split * run + run < n_units ? split * run + run : n_units;
    const int u_first = split * run + wave;   // this wave's units: u_first, + NW, ...
    const int nu = u_first < u_end ? (u_end - u_first + NW - 1) / NW : 0;

    const int lg = lane >> 4;                 // MFMA lane group
    const int ln = lane & 15;                 // MFMA row / column index
    // Token and head (of the KV head's group) of query row r, and this lane's last key + 1.
    auto row_token = [&](int r) { return PROMPT ? (int)((uint32_t)(row0 + r) / (uint32_t)G) : 0; };
    auto row_head = [&](int r) { return PROMPT ? row0 + r - row_token(r) * G : r; };
    auto q_row = [&](int r) { return PROMPT ? q_first + row_token(r) : (int64_t)seq; };
    const int my_keys = PROMPT ? pos0 + row_token(ln) + 1 : ctx;

    // ---- Q^T B operand: lane (lg, ln) takes head ln, 16-byte pieces 4 j + lg (zero for the
    // padding heads and dims). Issued before the block ids, whose wait covers it.
    u32x4 qf[KS];
#pragma unroll
    for (int j = 0; j < KS; ++j) {
        qf[j] = u32x4{0u, 0u, 0u, 0u};
        if (ln < rows && 4 * j + lg < CPR) {
            const Vec16 v = load16(reinterpret_cast<const char*>(p.q) +
                                   (q_row(ln) * p.q_st + (int64_t)(kvh * G + row_head(ln)) * p.q_sh) * ISZ +
                                   (4 * j + lg) * 16);
            qf[j] = u32x4{v.w[0], v.w[1], v.w[2], v.w[3]};
        }
    }

    // ---- fused append: the new token is the context's last key. The wave whose units end
    // with it holds the row (lanes 0 .. CPR-1 K, CPR .. 2 CPR-1 V) and stores it at the end.
    const int new_row = !PROMPT && p.app_slots && nu > 0 && u_first + (nu - 1) * NW == n_units - 1 ? (ctx - 1) % kUnit : -1;
    const char* knew = reinterpret_cast<const char*>(p.app_k) + ((int64_t)seq * p.app_st + (int64_t)kvh * p.app_sh) * ISZ;
    const char* vnew = reinterpret_cast<const char*>(p.app_v) + ((int64_t)seq * p.app_st + (int64_t)kvh * p.app_sh) * ISZ;
    Vec16 new_piece = Vec16{{0u, 0u, 0u, 0u}};
    int64_t new_slot = -1;
    static_assert(2 * CPR <= 64, "one piece per lane");
    if (new_row >= 0 && lane < 2 * CPR) {
        new_slot = p.app_slots[seq];
        new_piece = load16((lane < CPR ? knew : vnew) + (lane % CPR) * 16);
    }

    const int64_t slot_bytes = p.ss * ISZ;
    const int64_t block_bytes = p.sb * ISZ;
    const char* kbase = reinterpret_cast<const char*>(p.k) + (int64_t)kvh * p.sh * ISZ;
    const char* vbase = reinterpret_cast<const char*>(p.v) + (int64_t)kvh * p.sh * ISZ;
    const int64_t* table = p.tables + (int64_t)seq * p.table_stride;

    // ---- DMA of a unit: row and swizzled source chunk of this lane's instruction j.
    auto dma_row = [&](int j) { return (64 * j + lane) / CPR; };
    auto dma_chunk = [&](int j) { return (64 * j + lane) % CPR ^ C::swizzle((64 * j + lane) / CPR); };
    uint32_t lane_off[IPB];                   // inside an 8-row half
#pragma unroll
    for (int j = 0; j < IPB; ++j)
        lane_off[j] = (uint32_t)((dma_row(j) & 7) * slot_bytes) + (uint32_t)(dma_chunk(j) * 16);
    // offs: this lane's 8-key half's byte offset in the pool (half lane & 1 of the chunk's
    // unit lane / 2).
    auto dma_unit = [&](int k, int64_t offs, int slot) {
        const int64_t half0 = readlane64(offs, 2 * (k & 31)), half1 = readlane64(offs, 2 * (k & 31) + 1);
        const int unit = u_first + k * NW;
        const int rows = ctx - unit * kUnit < kUnit ? ctx - unit * kUnit : kUnit;   // keys of the unit
        const uint32_t lk = lds_addr(s_ring[wave][slot][0]), lv = lds_addr(s_ring[wave][slot][1]);
        const int app_row = unit == n_units - 1 ? new_row : -1;
        if (rows == kUnit && app_row < 0) {
#pragma unroll
            for (int j = 0; j < IPB; ++j) {
                if constexpr (kHalf) {
                    const int64_t half = 64 * j / CPR < 8 ? half0 : half1;
                    dma16_nt(kbase + half, lane_off[j], lk + j * 1024);
                    dma16_nt(vbase + half, lane_off[j], lv + j * 1024);
                } else if (kWhole || 64 * j + lane < kUnit * CPR) {
                    const int64_t off = (dma_row(j) < 8 ? half0 : half1) + lane_off[j];
                    dma16_nt(kbase + off, lk + j * 1024);
                    dma16_nt(vbase + off, lv + j * 1024);
                }
            }
            return;
        }
        // The context's last unit: rows past the context re-read its last key, the new
        // token's row comes from the caller (its pool slot is not read in this launch).
#pragma unroll
        for (int j = 0; j < IPB; ++j) {
            const int r = dma_row(j) < rows ? dma_row(j) : rows - 1;
            const int64_t off = (r < 8 ? half0 : half1) + (r & 7) * slot_bytes + dma_chunk(j) * 16;
            const char* ks = r == app_row ? knew + dma_chunk(j) * 16 : kbase + off;
            const char* vs = r == app_row ? vnew + dma_chunk(j) * 16 : vbase + off;
            if (kWhole || 64 * j + lane < kUnit * CPR) {
                dma16_nt(ks, lk + j * 1024);
                dma16_nt(vs, lv + j * 1024);
            }
        }
    };

    C unit;
    unit.address(lg, ln);
    f32x4 o[VT];
#pragma unroll
    for (int t = 0; t < VT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = kNegInf, l_part = 0.f;
    const float scale = p.scale;

    constexpr int kUnitDmas = 2 * IPB;
    for (int k0 = 0; k0 < nu; k0 += 32) {     // 32 units' block ids at a time
        int64_t offs;
        {
            int key = (u_first + (k0 + (lane >> 1)) * NW) * kUnit + 8 * (lane & 1);
            const int last = (ctx - 1) & ~7;
            key = key < last ? key : last;    // halves past the context: the last one's block
            const int64_t id = table[key >> p.block_shift];
            offs = ((uint64_t)id < (uint64_t)p.num_blocks ? id : 0) * block_bytes +
                   (key & (p.block_size - 1)) * slot_bytes;
        }
        const int k1 = k0 + 32 < nu ? k0 + 32 : nu;
        dma_unit(k0, offs, 0);
        if (k0 + 1 < k1) dma_unit(k0 + 1, offs, 1);
        for (int k = k0; k < k1; ++k) {
            const int slot = k & 1;
            if (k + 1 < k1) wait_vm<kUnitDmas>();
            else wait_vm<0>();
            unit.read(s_ring[wave][slot][0], s_ring[wave][slot][1], lg);
            if (k + 2 < k1) dma_unit(k + 2, offs, slot);

            // S^T for the 16 keys: lane (lg, ln) holds keys 4 lg + r of head ln.
            f32x4 st = unit.scores(qf);
            const int valid = my_keys - (u_first + k * NW) * kUnit;
            float bmax = kNegInf;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float x = C::scaled(st[r], scale);
                st[r] = 4 * lg + r < valid ? x : kNegInf;
                bmax = fmaxf(bmax, st[r]);
            }
            {
                SwapPair sp = swap16(bmax);
                bmax = fmaxf(sp.a, sp.b);
                sp = swap32(bmax);
                bmax = fmaxf(sp.a, sp.b);
            }
            const bool raise = bmax > m_run + kLazyMax;
            if (__builtin_amdgcn_ballot_w64(raise)) {
                const float m_new = raise ? bmax : m_run;
                const float alpha = !raise ? 1.f : (m_run == kNegInf ? 0.f : fast_exp2(m_run - m_new));
#pragma unroll
                for (int t = 0; t < VT; ++t) o[t] *= alpha;
                l_part *= alpha;
                m_run = m_new;
            }
            // Weights against the unit's own maximum, and what takes them to the running one.
            const float m_ref = sizeof(T) == 2 ? bmax : m_run;
            const float m_off = m_ref == kNegInf ? 0.f : m_ref;
            float pr[4], psum = 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pr[r] = fast_exp2(st[r] - m_off);
                psum += pr[r];
            }
            const float sc = sizeof(T) == 2 ? (bmax == kNegInf ? 0.f : fast_exp2(bmax - m_run)) : 1.f;
            l_part = fmaf(psum, sc, l_part);
            unit.accumulate(pr, sc, o);
        }
    }
    if (new_row >= 0 && (uint64_t)new_slot < (uint64_t)(p.num_blocks << p.block_shift)) {
        const int64_t dst = (new_slot >> p.block_shift) * block_bytes +
                            (new_slot & (p.block_size - 1)) * slot_bytes + (lane % CPR) * 16;
        store16(const_cast<char*>(lane < CPR ? kbase : vbase) + dst, new_piece);
    }

    // ---- the waves' partials over their own ring slices (no longer in use), then the merge.
    {
        SwapPair sp = swap16(l_part);
        l_part = sp.a + sp.b;
        sp = swap32(l_part);
        l_part = sp.a + sp.b;
    }
    float* w_acc = reinterpret_cast<float*>(s_ring[wave]);   // [G][D]
    if (ln < rows) {
#pragma unroll
        for (int t = 0; t < VT; ++t)
            *reinterpret_cast<float4*>(w_acc + ln * D + 16 * t + 4 * lg) = make_float4(o[t][0], o[t][1], o[t][2], o[t][3]);
        if (lg == 0) {
            s_ml[wave][ln][0] = m_run;
            s_ml[wave][ln][1] = l_part;
        }
    }
    lds_barrier();

    const int head0 = kvh * G;
    // Four consecutive elements per thread.
    const bool wide =
        (((uint64_t)(uintptr_t)p.out | (uint64_t)(p.out_st * ISZ) | (uint64_t)(p.out_sh * ISZ)) & (4 * ISZ - 1)) == 0;
    auto store_out = [&](int g, int d, float4 v) {
        T* orow = reinterpret_cast<T*>(p.out) + q_row(g) * p.out_st + (int64_t)(head0 + row_head(g)) * p.out_sh + d;
        C::store4(orow, v, wide);
    };
    for (int e = tid * 4; e < rows * D; e += NT * 4) {
        const int g = e / D, d = e - g * D;
        float M = kNegInf;
#pragma unroll
        for (int w = 0; w < NW; ++w) M = fmaxf(M, s_ml[w][g][0]);
        float L = 0.f;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float mw = s_ml[w][g][0];
            const float sc = mw == kNegInf ? 0.f : fast_exp2(mw - M);
            L += sc * s_ml[w][g][1];
            const float4 v = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(s_ring[w]) + e);
            acc.x += sc * v.x;
            acc.y += sc * v.y;
            acc.z += sc * v.z;
            acc.w += sc * v.w;
        }
        if (PROMPT || n_splits == 1) {
            const float inv = 1.f / L;
            store_out(g, d, make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv));
        } else {
            // Agent-scope stores: written through to where every XCD's agent-scope loads
            // read (the merging workgroup may run behind another L2).
            const int64_t slot = ((int64_t)seq * p.num_heads + head0 + g) * p.max_parts + split;
            const uint64_t lo = (uint64_t)__builtin_bit_cast(uint32_t, acc.y) << 32 | __builtin_bit_cast(uint32_t, acc.x);
            const uint64_t hi = (uint64_t)__builtin_bit_cast(uint32_t, acc.w) << 32 | __builtin_bit_cast(uint32_t, acc.z);
            uint64_t* po = reinterpret_cast<uint64_t*>(p.ws_o + slot * D + d);
            __hip_atomic_store(po, lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(po + 1, hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (d == 0) {
                const uint64_t ml = (uint64_t)__builtin_bit_cast(uint32_t, L) << 32 | __builtin_bit_cast(uint32_t, M);
                __hip_atomic_store(reinterpret_cast<uint64_t*>(p.ws_ml + slot * 2), ml, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    if (PROMPT || n_splits == 1) return;

    // ---- the last workgroup of the (sequence, KV head) to get here merges its runs, in run
    // order, and returns the counter to zero for the next call. The partial stores above are
    // performed before the counter moves: s_waitcnt vmcnt(0) holds the wave until each store
    // is acknowledged from the agent's coherence point, and the "memory" clobber keeps the
    // compiler from moving them past it. (No agent-scope release fence: it also writes back
    // the XCD's L2 and was measured to serialise the launch.)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    uint32_t* cnt = p.ws_cnt + ((int64_t)seq * KV + kvh);
    if (tid == 0) s_arrived = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (s_arrived != (uint32_t)(n_splits - 1)) return;
    if (tid == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    constexpr int CH = 8;                     // runs whose loads are in flight together
    for (int e = tid * 4; e < G * D; e += NT * 4) {
        const int g = e / D, d = e - g * D;
        const int64_t base = ((int64_t)seq * p.num_heads + head0 + g) * p.max_parts;
        uint64_t* ml = reinterpret_cast<uint64_t*>(p.ws_ml + base * 2);
        uint64_t* po = reinterpret_cast<uint64_t*>(p.ws_o + base * D + d);
        float M = kNegInf, L = 0.f;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int s0 = 0; s0 < n_splits; s0 += CH) {
            uint64_t mlv[CH], a[CH], b[CH];
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                const int s = s0 + j < n_splits ? s0 + j : n_splits - 1;
                mlv[j] = __hip_atomic_load(ml + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                a[j] = __hip_atomic_load(po + (int64_t)s * (D / 2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                b[j] = __hip_atomic_load(po + (int64_t)s * (D / 2) + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            auto lo = [](uint64_t x) { return __builtin_bit_cast(float, (uint32_t)x); };
            auto hi = [](uint64_t x) { return __builtin_bit_cast(float, (uint32_t)(x >> 32)); };
            float Mc = M;
#pragma unroll
            for (int j = 0; j < CH; ++j) Mc = fmaxf(Mc, lo(mlv[j]));
            const float rs = M == kNegInf ? 0.f : fast_exp2(M - Mc);
            L *= rs;
            acc.x *= rs;
            acc.y *= rs;
            acc.z *= rs;
            acc.w *= rs;
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                const float mj = lo(mlv[j]);
                const float sc = s0 + j >= n_splits || mj == kNegInf ? 0.f : fast_exp2(mj - Mc);
                if (s0 + j < n_splits) {
                    L += sc * hi(mlv[j]);
                    acc.x += sc * lo(a[j]);
                    acc.y += sc * hi(a[j]);
                    acc.z += sc * lo(b[j]);
                    acc.w += sc * hi(b[j]);
                }
            }
            M = Mc;
        }
        const float inv = 1.f / L;
        store_out(g, d, make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv));
    }
}

// Workgroups of NW waves for one (sequence, KV head) run each.
template <typename T, int D, int NW>
int launch_nw(const AttnParams& p, hipStream_t stream) {
    const int64_t pairs = (int64_t)p.num_seqs * p.num_kv_heads;
    const int64_t fits = (int64_t)kCus * wgs_per_cu(D * (int)sizeof(T), NW);
    const int64_t units = (int64_t)p.max_parts * (kDecodePart / kUnit);   // longest context's bound
    Cut cut{};
    // Units a wave that a run has at least (and a workspace slot's tokens), and that a context
    // may have before it is worth the merge: 2 and 4 where a unit is dear, fp32 products and
    // rows of 160 bytes up, else 3 and 8. Replayed from graphs, us a call, 2 and 4 vs 4 and 8:
    // 32/8 heads of 128, bf16, 4 sequences of 16-1000 tokens 9.9 vs 13.6, 16 of them 11.1 vs
    // 14.8; fp32, 16/4 heads of 64, 8 of 16-1000 9.6 vs 16.5. Over 40 batches of 1-64 sequences
    // of 300-8000 tokens (geometric means, relative), 2 and 4 / 3 and 6 / 3 and 8: 8/4 heads of
    // 80 0.93 / 0.94 / 1.01, 16/4 of 96 0.95 / 0.97 / 1.02, 12 heads of 64, fp16, 1.02 / 1.01 /
    // 1.03, 8/4 of 64 1.04 / 1.03 / 1.04; but a step captured for GPT-2's 1024 positions is
    // told of no longer context than 8 units a wave and spares the search at that bound (12
    // layers of 8 sequences 161 vs 166 us with 6).
    constexpr bool kDear = sizeof(T) == 4 || D >= 80;
    cut.min_run = NW * (kDear ? 2 : 3) > kDecodePart / kUnit ? NW * (kDear ? 2 : 3) : kDecodePart / kUnit;
    cut.whole = NW * (kDear ? 4 : 8);
    // Where the pairs fill the GPU by themselves, or the scan does not reach, contexts of less
    // than 32 units a wave are not cut; none are where the counters do not reach.
    cut.long_from = NW * 32;
    // (Up to 2^30 units a batch: the search's run, which starts there where none is cut, then
    // ends at once and stays far inside 32 bits.)
    const bool can = p.ws_cnt && p.num_seqs * units <= ((int64_t)1 << 30);
    if (can && p.num_seqs <= kMaxScanSeqs) {
        // Many pairs of long contexts: runs for two rounds, or the longest context would be
        // walked whole (250 sequences of 512-8192 tokens, 8/2 heads, bf16: 219 -> 189 us; 60 of
        // 16-2000, 12 heads of 64, fp32: 84 -> 72); with less to read the second round's start and
        // merges cost more than it evens out (64 of 16-2048, 12 heads of 64, fp16: 24 -> 25.5;
        // 120 of 1-1000, 32/8 heads, fp16: 49 -> 55).
        int64_t from = 0x7fffffff;
        if (2 * pairs > fits) from = ((int64_t)1 << 30) / (pairs * kUnit * D * 2 * (int64_t)sizeof(T)) + 1;
        if (pairs >= fits && from > 24 * NW) from = 24 * NW;
        cut.slots2_from = (int)from;
        cut.slots = pairs < fits ? (int)(fits / p.num_kv_heads) : 0;
        cut.slots2 = pairs < 2 * fits ? (int)(2 * fits / p.num_kv_heads) : 0;
    }
    const int slots = units >= cut.slots2_from ? cut.slots2 : cut.slots;
    int64_t grid = pairs;
    if (units > cut.whole && slots > 0) {
        cut.mode = kCutRuns;
        grid = (int64_t)(slots > p.num_seqs ? slots : p.num_seqs) * p.num_kv_heads;
    } else if (can && units >= cut.long_from && cut.slots == 0 && cut.slots2 == 0) {
        cut.mode = kCutLong;
        cut.slots = (int)(fits / p.num_kv_heads > 1 ? fits / p.num_kv_heads : 1);
        cut.min_run = cut.long_from / 2;
        grid = ((int64_t)p.num_seqs + cut.slots / 2) * p.num_kv_heads;
    }
    if (grid > 0x7fffffff) return PKV_EUNSUPPORTED;
    paged_decode_split_kernel<T, D, NW, false><<<dim3((unsigned)grid), NW * 64, 0, stream>>>(p, cut);
    return check_launch("paged decode attention (split)");
}

// Waves per workgroup: 8 while the pairs fit the GPU so (each context is walked by more
// waves: fewer splits, shorter chains), else 4. Measured, us a call, 8 vs 4 waves: 8
// sequences of 1-8k, 32/8 heads of 128, bf16 35.3 vs 37.5; 30 x 4096 82 vs 88; 64 sequences
// of 16-2048, 12 heads of 64, fp16 (768 pairs, more than fit) 25.2 vs 21.9. 2 where there
// are many rounds of pairs, whose starts and merges then overlap (4 vs 2 waves): 1000 of 1-60,
// 32/8 heads, bf16 69.8 vs 42.6; 300 of 1-120 26.9 vs 20.4; 400 of 1-60, 12 heads of 64 22.0
// vs 16.9; 200 of 1-100 (2.3 rounds) 16.2 vs 16.4;
// 128 of 512-4096, 32/8 heads of 128, fp32 418 vs 483: short contexts only. 16 waves were never better than 8 by more than the noise, but
// for 500 single-head sequences of 16-4000 (51 vs 58).
template <typename T, int D>
int launch_d(const AttnParams& p, hipStream_t stream) {
    const int64_t pairs = (int64_t)p.num_seqs * p.num_kv_heads;
    if constexpr (wgs_per_cu(D * (int)sizeof(T), 8) > 0)
        if (pairs <= (int64_t)kCus * wgs_per_cu(D * (int)sizeof(T), 8)) return launch_nw<T, D, 8>(p, stream);
    if (pairs >= 4ll * kCus * wgs_per_cu(D * (int)sizeof(T), 4) && p.max_parts * (kDecodePart / kUnit) <= 32)
        return launch_nw<T, D, 2>(p, stream);
    return launch_nw<T, D, 4>(p, stream);
}

template <typename T>
int launch_t(const AttnParams& p, hipStream_t stream) {
    switch (p.head_dim) {
        case 32: return launch_d<T, 32>(p, stream);
        case 48: return launch_d<T, 48>(p, stream);
        case 64: return launch_d<T, 64>(p, stream);
        case 80: return launch_d<T, 80>(p, stream);
        case 96: return launch_d<T, 96>(p, stream);
        case 112: return launch_d<T, 112>(p, stream);
        case 128: return launch_d<T, 128>(p, stream);
    }
    return PKV_EUNSUPPORTED;
}

// Row tiles of one KV head's batch at most (a sequence's last tile may be partial).
int64_t prompt_tiles(const AttnParams& p) { return p.num_tokens * p.group / kUnit + p.num_seqs; }

template <int D>
int launch_prompt(const AttnParams& p, hipStream_t stream) {
    const unsigned grid = (unsigned)(prompt_tiles(p) * p.num_kv_heads);
    paged_decode_split_kernel<float, D, 4, true><<<dim3(grid), 256, 0, stream>>>(p, Cut{});
    return check_launch("paged prompt attention (split)");
}

}  // namespace

// What both forms of the kernel ask of a batch.
static bool split_shape(const AttnParams& p, int dtype) {
    const int isz = dtype == PKV_FLOAT32 ? 4 : 2;
    if (p.num_blocks < 1 || p.block_shift < 3) return false;
    if (p.head_dim % 16 || p.head_dim < 32 || p.head_dim > 128) return false;
    // Units of a sequence are exact in fp32 (the run search divides in it).
    if ((int64_t)p.max_parts * kDecodePart >= ((int64_t)1 << 28)) return false;
    if (!slot_offsets_fit(p, 8, isz)) return false;   // inside an 8-row half
    // 16-byte rows, those of a fused append among them.
    uint64_t probe = (uint64_t)(uintptr_t)p.q | (uint64_t)(uintptr_t)p.k | (uint64_t)(uintptr_t)p.v |
                     (uint64_t)(p.q_st * isz) | (uint64_t)(p.q_sh * isz) | (uint64_t)(p.sb * isz) |
                     (uint64_t)(p.ss * isz) | (uint64_t)(p.sh * isz);
    if (p.app_slots)
        probe |= (uint64_t)(uintptr_t)p.app_k | (uint64_t)(uintptr_t)p.app_v | (uint64_t)(p.app_st * isz) |
                 (uint64_t)(p.app_sh * isz);
    return probe % 16 == 0;
}

bool decode_split_applies(const AttnParams& p, int dtype) {
    if (p.group > 16 || (int64_t)p.num_seqs * p.num_kv_heads > 0x7fffffff) return false;
    if (p.max_parts > 1 && (!p.ws_o || !p.ws_ml)) return false;
    return split_shape(p, dtype);
}

bool prompt_split_f32_applies(const AttnParams& p) {
    if (!p.qsl || p.app_slots || p.num_seqs > kMaxScanSeqs) return false;
    if (((int64_t)p.num_tokens + kUnit) * p.group > 0x7fffffff || prompt_tiles(p) * p.num_kv_heads > 0x7fffffff)
        return false;
    return split_shape(p, PKV_FLOAT32);
}

bool prompt_split_f32_few(const AttnParams& p) {
    const int per_cu = (160 * 1024) / (4 * 2 * 2 * kUnit * p.head_dim * 4 + 4 * 128 + 16);
    return p.num_tokens * p.num_heads / kUnit * 4 <= 9ll * kCus * (per_cu < 4 ? per_cu : 4);
}

int launch_prompt_split_f32(const AttnParams& p, hipStream_t stream) {
    if (!prompt_split_f32_applies(p)) return PKV_EUNSUPPORTED;
    switch (p.head_dim) {
        case 32: return launch_prompt<32>(p, stream);
        case 48: return launch_prompt<48>(p, stream);
        case 64: return launch_prompt<64>(p, stream);
        case 80: return launch_prompt<80>(p, stream);
        case 96: return launch_prompt<96>(p, stream);
        case 112: return launch_prompt<112>(p, stream);
        case 128: return launch_prompt<128>(p, stream);
    }
    return PKV_EUNSUPPORTED;
}

int launch_decode_split(const AttnParams& p, int dtype, hipStream_t stream) {
    if (!decode_split_applies(p, dtype)) return PKV_EUNSUPPORTED;
    if (p.num_seqs == 0) return PKV_OK;
    if (dtype == PKV_FLOAT32) return launch_t<float>(p, stream);
    return dtype == PKV_FLOAT16 ? launch_t<_Float16>(p, stream) : launch_t<bf16_t>(p, stream);
}

}  // namespace pkv
