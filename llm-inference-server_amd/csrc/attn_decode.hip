// Paged decode attention for fp32 pools, block_size 16, head_dim 64, one or two query heads per
// KV head: a partition kernel with K/V staged in registers, and a split-KV merge kernel.
//
// Bound: HBM and the arithmetic beside it. With so few heads a group the one-launch MFMA kernel
// (attn_decode_split.hip) spends its fp32 matrix steps on 16 columns of which one or two count;
// here each product is computed once. Measured, us a call replayed from a graph, this kernel
// first, 12 heads: 8 sequences of 16-500 tokens 8.3 vs 11.3, 16 of 500-1000 18.2 vs 20.7, 32 of
// 16-1000 22.7 vs 23.7, 64 of 200-3000 114 vs 129, 22 of 16-1000 18.8 vs 18.8; issued eagerly
// its second launch can cost the host more than that (22 of 16-1000 with the append 24.7 vs
// 22.8), but a rule on sizes would have an eager step and its captured form, which is told the
// longest context its tables allow, run different kernels. Groups of 2, 6 KV heads: 64 of
// 500-2000 46 vs 57; of 4 the other is even or faster (8 of 16-1000 10.7 vs 9.6), of 8 faster
// (200 of 500-2000 68 vs 61).
//
//  * Work unit = (KV head, 256-token partition, sequence): one 256-thread workgroup of 4
//    wave64s, 64 tokens (4 blocks) per wave.
//  * Latency chain per wave: ONE vector load of the wave's 4 block-table entries (broadcast
//    with readlane), then all K loads of the 4 blocks at once, the scores, then all V loads
//    at once, issued before the softmax so they are in flight while it runs.
//  * Split-KV: a sequence that fits one partition is finished in place; otherwise each
//    partition writes its partial (max, denominator, unnormalised output) and the second
//    kernel on the same stream merges them with the log-sum-exp rule.
// Keys at or beyond context_lens are never loaded.
#include <type_traits>

#include "attention.h"

namespace pkv {
namespace {

constexpr int kBS = 16;
constexpr int kWaves = kDecodePart / 64;  // 64 tokens per wave
constexpr int kTPW = 64;
constexpr int kBPW = kTPW / kBS;          // blocks per wave

// Partial dot product of one 16-byte chunk of K with the matching chunk of q.
__device__ __forceinline__ float chunk_dot(const Vec16& k, const Vec16& q, float acc) {
#pragma unroll
    for (int w = 0; w < 4; ++w)
        acc = fmaf(__builtin_bit_cast(float, k.w[w]), __builtin_bit_cast(float, q.w[w]), acc);
    return acc;
}

// K/V rows are read exactly once per launch: streaming loads.
__device__ __forceinline__ Vec16 kv_load16(const void* ptr) { return load16_stream(ptr); }
__device__ __forceinline__ uint2 kv_load8(const void* ptr) { return load8_stream(ptr); }

template <int D, int G>
__global__ __launch_bounds__(kWaves * 64) void paged_decode_kernel(const AttnParams p) {
    using T = float;
    constexpr int ISZ = (int)sizeof(T);
    constexpr int CHUNKS = D * ISZ / 16;      // K: 16-byte chunks per (token, head) row
    constexpr int KLPT = 8;                   // K: lanes per token (8 x 16 B = one 128-byte line)
    constexpr int CPL = CHUNKS / KLPT;        // K: chunks per lane
    constexpr int KGRP = kBS * KLPT / 64;     // K: load groups per block (8 tokens each)
    constexpr int EPV = 8 / ISZ;              // V: elements per 8-byte chunk
    constexpr int VLPT = D * ISZ / 8;         // V: lanes per token
    constexpr int TSV = 64 / VLPT;            // V: tokens per load step
    constexpr int VSTEPS = kTPW / TSV;        // V: load steps per wave
    static_assert(CHUNKS % KLPT == 0 && G <= KLPT && 64 % VLPT == 0 && kBS % TSV == 0 && VSTEPS % 2 == 0,
                  "unsupported head_dim / group");

    __shared__ float s_p[kWaves][kTPW][G];    // scores, then probabilities
    __shared__ float s_acc[kWaves][G][D];
    __shared__ float s_ml[kWaves][G][2];

    const int kvh = (int)blockIdx.x;
    const int part = (int)blockIdx.y;
    const int seq = (int)blockIdx.z;
    // Memory safety for out-of-contract input: never walk past the table row or the
    // partitions the grid/workspace were sized for (the host guarantees neither
    // bound binds for valid input).
    int64_t ctx64 = p.ctx_lens[seq];
    ctx64 = ctx64 < (int64_t)p.table_width * kBS ? ctx64 : (int64_t)p.table_width * kBS;
    ctx64 = ctx64 < (int64_t)p.max_parts * kDecodePart ? ctx64 : (int64_t)p.max_parts * kDecodePart;
    const int ctx = (int)ctx64;
    const int part_start = part * kDecodePart;
    if (part_start >= ctx) return;
    const int n_parts = (ctx + kDecodePart - 1) / kDecodePart;

    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wstart = part_start + wave * kTPW;  // multiple of 16
    const char* kbase = reinterpret_cast<const char*>(p.k) + (int64_t)kvh * p.sh * ISZ;
    const char* vbase = reinterpret_cast<const char*>(p.v) + (int64_t)kvh * p.sh * ISZ;
    const uint32_t slot_bytes = (uint32_t)(p.ss * ISZ);
    const int64_t block_bytes = p.sb * ISZ;

    // ------------------------------------------------------------ block ids + q
    // Lane b < kBPW fetches the wave's b-th block id; -1 marks "beyond the context"
    // and ids outside the pool are treated the same way (never dereferenced).
    int64_t my_blk = -1;
    if (lane < kBPW && wstart + lane * kBS < ctx)
        my_blk = p.tables[(int64_t)seq * p.table_stride + wstart / kBS + lane];
    const int kj = lane % KLPT;   // which 16-byte chunks of the row: kj, kj + 8, ...
    const int ktok = lane / KLPT; // token within a load group
    Vec16 q[G][CPL];
    {
        const char* qrow = reinterpret_cast<const char*>(p.q) + ((int64_t)seq * p.q_st + (int64_t)kvh * G * p.q_sh) * ISZ;
        const int64_t q_head_bytes = p.q_sh * ISZ;
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int i = 0; i < CPL; ++i) q[g][i] = load16(qrow + g * q_head_bytes + (i * KLPT + kj) * 16);
    }
    const char* kblk[kBPW];
    const char* vblk[kBPW];
    bool live[kBPW];
#pragma unroll
    for (int b = 0; b < kBPW; ++b) {
        const int64_t id = readlane64(my_blk, b);
        live[b] = (uint64_t)id < (uint64_t)p.num_blocks;
        kblk[b] = kbase + id * block_bytes;
        vblk[b] = vbase + id * block_bytes;
    }

    // ------------------------------------------------------------ K, scores, V issue
    // Fast path (wave-uniform): all 64 tokens inside the context and all 4 block ids
    // inside the pool. Its loads are unconditional and nothing is zero-filled; the other
    // waves (at most the last two of a sequence) predicate every load and zero what they
    // skip, which costs ~15% more VALU instructions.
    bool full = wstart + kTPW <= ctx;
#pragma unroll
    for (int b = 0; b < kBPW; ++b) full = full && live[b];
    // K: each load instruction reads 8 tokens x one whole 128-byte line of their rows.
    const uint32_t k_lane_off = ktok * slot_bytes + (uint32_t)(kj * 16);
    const int vchunk = lane % VLPT;
    const int vslot = lane / VLPT;
    Vec16 kv[kBPW][KGRP][CPL];
    uint2 vv[VSTEPS];
    auto stream = [&](auto full_tag) {
        constexpr bool FULL = decltype(full_tag)::value;
#pragma unroll
        for (int b = 0; b < kBPW; ++b)
#pragma unroll
            for (int gr = 0; gr < KGRP; ++gr) {
                if (FULL || live[b]) {
#pragma unroll
                    for (int i = 0; i < CPL; ++i)
                        kv[b][gr][i] = kv_load16(kblk[b] + (k_lane_off + (uint32_t)(gr * 8) * slot_bytes +
                                                            (uint32_t)(i * KLPT * 16)));
                } else {
#pragma unroll
                    for (int i = 0; i < CPL; ++i) kv[b][gr][i] = Vec16{{0u, 0u, 0u, 0u}};
                }
            }
#pragma unroll
        for (int b = 0; b < kBPW; ++b)
#pragma unroll
            for (int gr = 0; gr < KGRP; ++gr) {
                const int t_rel = b * kBS + gr * 8 + ktok;
                const bool valid = FULL || (live[b] && wstart + t_rel < ctx);
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    float s = 0.f;
#pragma unroll
                    for (int i = 0; i < CPL; ++i) s = chunk_dot(kv[b][gr][i], q[g][i], s);
                    s = ref_score_log2<T>(octet_sum(s), p.scale);
                    if (g == kj) s_p[wave][t_rel][g] = valid ? s : kNegInf;
                }
            }
        // V: issued before the softmax so the loads are in flight while it runs.
#pragma unroll
        for (int st = 0; st < VSTEPS; ++st) {
            const int b = (st * TSV) / kBS;
            const int t_rel = st * TSV + vslot;
            const uint32_t off = (uint32_t)(t_rel % kBS) * slot_bytes + (uint32_t)(vchunk * 8);
            if (FULL) {
                vv[st] = kv_load8(vblk[b] + off);
            } else {
                vv[st] = make_uint2(0u, 0u);
                if (live[b] && wstart + t_rel < ctx) vv[st] = kv_load8(vblk[b] + off);
            }
        }
    };
    if (full) stream(std::true_type{});
    else stream(std::false_type{});
    // Scores, softmax and P·V stay inside the wave's own slice of s_p, so the waves only
    // order their own LDS traffic here; the workgroup meets once, at the merge.
    wave_lds_sync();

    // ------------------------------------------------------------ softmax (lane = token)
    float m_w[G], l_w[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const float a = s_p[wave][lane][g];
        const float m = wave_max(a);
        const float pr = m == kNegInf ? 0.f : fast_exp2(a - m);
        s_p[wave][lane][g] = pr;
        m_w[g] = m;
        l_w[g] = wave_sum(pr);
    }
    wave_lds_sync();

    // ------------------------------------------------------------ P·V
    float acc[G][EPV];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int e = 0; e < EPV; ++e) acc[g][e] = 0.f;
#pragma unroll
    for (int st = 0; st < VSTEPS; ++st) {
        const int t_rel = st * TSV + vslot;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const float pg = s_p[wave][t_rel][g];
            acc[g][0] = fmaf(pg, __builtin_bit_cast(float, vv[st].x), acc[g][0]);
            acc[g][1] = fmaf(pg, __builtin_bit_cast(float, vv[st].y), acc[g][1]);
        }
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int e = 0; e < EPV; ++e) acc[g][e] = fold_lanes<VLPT>(acc[g][e]);
    if (vslot == 0) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < EPV; ++e) s_acc[wave][g][vchunk * EPV + e] = acc[g][e];
    }
    if (lane == 0) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            s_ml[wave][g][0] = m_w[g];
            s_ml[wave][g][1] = l_w[g];
        }
    }
    lds_barrier();

    // ------------------------------------------------------------ merge the waves
    const int head0 = kvh * G;
    for (int idx = (int)threadIdx.x; idx < G * D; idx += kWaves * 64) {
        const int g = idx / D, d = idx - g * D;
        float M = kNegInf;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) M = fmaxf(M, s_ml[w][g][0]);
        float L = 0.f, O = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float mw = s_ml[w][g][0];
            const float sc = mw == kNegInf ? 0.f : fast_exp2(mw - M);
            L += sc * s_ml[w][g][1];
            O += sc * s_acc[w][g][d];
        }
        if (n_parts == 1) {
            T* orow = reinterpret_cast<T*>(p.out) + (int64_t)seq * p.out_st + (int64_t)(head0 + g) * p.out_sh;
            orow[d] = from_f32<T>(O / L);
        } else {
            const int64_t slot = ((int64_t)seq * p.num_heads + head0 + g) * p.max_parts + part;
            p.ws_o[slot * D + d] = O;
            if (d == 0) {
                p.ws_ml[slot * 2] = M;
                p.ws_ml[slot * 2 + 1] = L;
            }
        }
    }
}

// Split-KV merge, launched after the partition kernel on the same stream (stream
// order is the only synchronisation: no fences, no atomics). One workgroup per
// (KV head, sequence) merges the partitions' (max, denominator, output) with the
// log-sum-exp rule; sequences that fit one PART-token partition were finished by the
// partition kernel and are skipped.
// Threads of a merge workgroup: the G * D / 2 element pairs of one KV head, in whole
// waves, at most 256 (one wave for a head_dim-64 group of one).
template <int G, int D>
constexpr int kCombineThreads = (G * D / 2 + 63) / 64 * 64 < 256 ? (G * D / 2 + 63) / 64 * 64 : 256;

template <int D, int G>
__global__ __launch_bounds__((kCombineThreads<G, D>)) void paged_decode_combine_kernel(const AttnParams p) {
    using T = float;
    constexpr int PART = kDecodePart;
    const int kvh = (int)blockIdx.x;
    const int seq = (int)blockIdx.y;
    int64_t ctx64 = p.ctx_lens[seq];
    ctx64 = ctx64 < (int64_t)p.table_width * kBS ? ctx64 : (int64_t)p.table_width * kBS;
    ctx64 = ctx64 < (int64_t)p.max_parts * kDecodePart ? ctx64 : (int64_t)p.max_parts * kDecodePart;
    const int n_parts = (int)((ctx64 + PART - 1) / PART);
    if (n_parts <= 1) return;
    const int head0 = kvh * G;
    constexpr int CH = 16;  // partitions whose loads are in flight together
    static_assert(D % 2 == 0, "pairs of head_dim elements");
    // Each thread merges two adjacent head_dim elements (8-byte loads), so G * D <= 512
    // (every shape the partition kernels take) is one pass of dependent loads.
    for (int idx = (int)threadIdx.x; idx < G * D / 2; idx += kCombineThreads<G, D>) {
        const int g = (2 * idx) / D, d = 2 * idx - g * D;
        const int64_t base = ((int64_t)seq * p.num_heads + head0 + g) * p.max_parts;
        const float2* ml = reinterpret_cast<const float2*>(p.ws_ml) + base;
        const float2* o = reinterpret_cast<const float2*>(p.ws_o + base * D + d);
        // Online log-sum-exp over the partitions, CH at a time.
        float M = kNegInf, L = 0.f, O0 = 0.f, O1 = 0.f;
        for (int pt0 = 0; pt0 < n_parts; pt0 += CH) {
            float2 mlv[CH], ov[CH];
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                const bool in = pt0 + j < n_parts;
                mlv[j] = in ? ml[pt0 + j] : make_float2(kNegInf, 0.f);
                ov[j] = in ? o[(int64_t)(pt0 + j) * (D / 2)] : make_float2(0.f, 0.f);
            }
            float Mc = M;
#pragma unroll
            for (int j = 0; j < CH; ++j) Mc = fmaxf(Mc, mlv[j].x);
            const float rescale = M == kNegInf ? 0.f : fast_exp2(M - Mc);
            L *= rescale;
            O0 *= rescale;
            O1 *= rescale;
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                const float sc = mlv[j].x == kNegInf ? 0.f : fast_exp2(mlv[j].x - Mc);
                L += sc * mlv[j].y;
                O0 += sc * ov[j].x;
                O1 += sc * ov[j].y;
            }
            M = Mc;
        }
        T* orow = reinterpret_cast<T*>(p.out) + (int64_t)seq * p.out_st + (int64_t)(head0 + g) * p.out_sh;
        orow[d] = from_f32<T>(O0 / L);
        orow[d + 1] = from_f32<T>(O1 / L);
    }
}

template <int D, int G>
int launch_g(const AttnParams& p, dim3 grid, hipStream_t stream) {
    paged_decode_kernel<D, G><<<grid, kWaves * 64, 0, stream>>>(p);
    int rc = check_launch("paged decode attention");
    if (rc || p.max_parts == 1) return rc;
    paged_decode_combine_kernel<D, G><<<dim3(grid.x, grid.z), kCombineThreads<G, D>, 0, stream>>>(p);
    return check_launch("paged decode combine");
}

}  // namespace

bool decode_f32_applies(const AttnParams& p) {
    if (p.block_size != kBS || p.head_dim != 64 || (p.group != 1 && p.group != 2)) return false;
    if (p.num_kv_heads > 65535 || p.max_parts > 65535 || p.num_seqs > 65535) return false;
    if (p.max_parts > 1 && (!p.ws_o || !p.ws_ml)) return false;
    if (!slot_offsets_fit(p, kBS, 4)) return false;
    // 16-byte chunk loads need 16-byte aligned rows.
    const uint64_t probe = (uint64_t)(uintptr_t)p.q | (uint64_t)(uintptr_t)p.k | (uint64_t)(uintptr_t)p.v |
                           (uint64_t)(p.q_st * 4) | (uint64_t)(p.q_sh * 4) | (uint64_t)(p.sb * 4) |
                           (uint64_t)(p.ss * 4) | (uint64_t)(p.sh * 4);
    return probe % 16 == 0;
}

int launch_decode_f32(const AttnParams& p, hipStream_t stream) {
    if (!decode_f32_applies(p)) return PKV_EUNSUPPORTED;
    const dim3 grid((unsigned)p.num_kv_heads, (unsigned)p.max_parts, (unsigned)p.num_seqs);
    return p.group == 1 ? launch_g<64, 1>(p, grid, stream) : launch_g<64, 2>(p, grid, stream);
}

}  // namespace pkv
