// Paged decode attention for fp32 pools, block_size 16, head_dim 64, one or two query heads per
// KV head: a partition kernel with K/V staged in registers, which appends the new rows and
// merges the partitions itself or, in large batches, leaves both to launches of their own.
//
// Bound: HBM and the arithmetic beside it, the start and the merge in small batches. With so few
// heads a group the one-launch MFMA kernel (attn_decode_split.hip) spends its fp32 matrix steps
// on 16 columns of which one or two count; here each product is computed once. Measured, us a
// call replayed from a graph, this kernel first, 12 heads: 8 sequences of 16-500 tokens 8.4 vs
// 14.2, 16 of 500-1000 17.4 vs 22.8, 22 of 16-1000 19.4 vs 22.9, 64 of 200-3000 106 vs 129.
// Groups of 2, 6 KV heads: 64 of 500-2000 48 vs 59; of 4 the other is even or faster (8 of
// 16-1000 10.7 vs 9.6), of 8 faster (200 of 500-2000 68 vs 61). A rule on sizes would have an
// eager step and its captured form, which is told the longest context its tables allow, run
// different kernels.
//
//  * Work unit = (KV head, 256-token partition, sequence): one 256-thread workgroup of 4
//    wave64s, 64 tokens (4 blocks) per wave.
//  * Latency chain per wave: ONE vector load of the wave's 4 block-table entries (broadcast
//    with readlane), then all K loads of the 4 blocks at once, the scores, then all V loads
//    at once, issued before the softmax so they are in flight while it runs.
//  * Split-KV: a sequence that fits one partition is finished in place; otherwise each
//    partition writes its partial (max, denominator, unnormalised output), and the last
//    workgroup of the (sequence, KV head) to end, or a second kernel on the same stream, merges
//    them in order with the log-sum-exp rule.
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

// A pair of a partial. FUSED: agent-scope accesses, written through to where every XCD's
// agent-scope loads read (the merging workgroup may run behind another L2); else another
// launch reads what one wrote.
template <bool FUSED>
__device__ __forceinline__ void put_pair(float* at, float x, float y) {
    uint64_t* to = reinterpret_cast<uint64_t*>(at);
    const uint64_t v = (uint64_t)__builtin_bit_cast(uint32_t, y) << 32 | __builtin_bit_cast(uint32_t, x);
    if constexpr (FUSED) __hip_atomic_store(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *to = v;
}
template <bool FUSED>
__device__ __forceinline__ float2 get_pair(float* at) {
    uint64_t* from = reinterpret_cast<uint64_t*>(at);
    uint64_t v;
    if constexpr (FUSED) v = __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else v = *from;
    return make_float2(__builtin_bit_cast(float, (uint32_t)v), __builtin_bit_cast(float, (uint32_t)(v >> 32)));
}

// Merge of a (KV head, sequence)'s partitions by one wave, each lane two adjacent head_dim
// elements of one head: the online log-sum-exp rule over them in order, CH at a time.
template <int D, int G, bool FUSED>
__device__ __forceinline__ void merge_partitions(const AttnParams& p, int seq, int kvh, int n_parts) {
    constexpr int CH = 16;                    // partitions whose loads are in flight together
    static_assert(D % 2 == 0 && G * D / 2 <= 64, "one wave");
    const int lane = lane_id();
    if (lane >= G * D / 2) return;
    const int head = kvh * G + 2 * lane / D, d = 2 * lane % D;
    const int64_t base = ((int64_t)seq * p.num_heads + head) * p.max_parts;
    float* ml = p.ws_ml + base * 2;
    float* o = p.ws_o + base * D + d;
    float M = kNegInf, L = 0.f, O0 = 0.f, O1 = 0.f;
    for (int pt0 = 0; pt0 < n_parts; pt0 += CH) {
        float2 mlv[CH], ov[CH];
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const bool in = pt0 + j < n_parts;
            mlv[j] = in ? get_pair<FUSED>(ml + (pt0 + j) * 2) : make_float2(kNegInf, 0.f);
            ov[j] = in ? get_pair<FUSED>(o + (int64_t)(pt0 + j) * D) : make_float2(0.f, 0.f);
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
    float* orow = reinterpret_cast<float*>(p.out) + (int64_t)seq * p.out_st + (int64_t)head * p.out_sh;
    orow[d] = O0 / L;
    orow[d + 1] = O1 / L;
}

template <int D, int G, bool FUSED>
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

    // ------------------------------------------------------------ fused append
    // The new token is the context's last key: the wave that holds it takes its row from the
    // caller (its pool slot is not read in this launch) and stores it, lanes 0 .. CHUNKS-1 the
    // K row, CHUNKS .. 2 CHUNKS-1 the V row.
    const bool has_new = FUSED && p.app_slots && ctx - 1 >= wstart && ctx - 1 < wstart + kTPW;
    const int new_tok = has_new ? ctx - 1 - wstart : -1;
    const char* knew = reinterpret_cast<const char*>(p.app_k) + ((int64_t)seq * p.app_st + (int64_t)kvh * p.app_sh) * ISZ;
    const char* vnew = reinterpret_cast<const char*>(p.app_v) + ((int64_t)seq * p.app_st + (int64_t)kvh * p.app_sh) * ISZ;
    static_assert(2 * CHUNKS <= 64, "one piece per lane");
    Vec16 new_piece = Vec16{{0u, 0u, 0u, 0u}};
    int64_t new_slot = -1;
    if (has_new && lane < 2 * CHUNKS) {
        new_slot = p.app_slots[seq];
        new_piece = load16((lane < CHUNKS ? knew : vnew) + lane % CHUNKS * 16);
    }

    // ------------------------------------------------------------ K, scores, V issue
    // Fast path (wave-uniform): all 64 tokens inside the context and in the pool, all 4 block
    // ids inside it. Its loads are unconditional and nothing is zero-filled; the other
    // waves (at most the last two of a sequence) predicate every load and zero what they
    // skip, which costs ~15% more VALU instructions.
    bool full = wstart + kTPW <= ctx && !has_new;
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
                    const char* row = kblk[b] + (k_lane_off + (uint32_t)(gr * 8) * slot_bytes);
                    if (!FULL && b * kBS + gr * 8 + ktok == new_tok) row = knew + kj * 16;
#pragma unroll
                    for (int i = 0; i < CPL; ++i) kv[b][gr][i] = kv_load16(row + i * KLPT * 16);
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
                if (live[b] && wstart + t_rel < ctx)
                    vv[st] = kv_load8(t_rel == new_tok ? vnew + vchunk * 8 : vblk[b] + off);
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
    if (has_new && (uint64_t)new_slot < (uint64_t)p.num_blocks * kBS) {
        const int64_t dst = new_slot / kBS * block_bytes + new_slot % kBS * (int64_t)slot_bytes + lane % CHUNKS * 16;
        store16(const_cast<char*>(lane < CHUNKS ? kbase : vbase) + dst, new_piece);
    }
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
    // In the first wave, two adjacent head_dim elements a lane.
    if (wave != 0) return;
    static_assert(G * D / 2 <= 64, "one wave");
    if (lane < G * D / 2) {
        const int g = 2 * lane / D, d = 2 * lane % D;
        float M = kNegInf;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) M = fmaxf(M, s_ml[w][g][0]);
        float L = 0.f, O0 = 0.f, O1 = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float mw = s_ml[w][g][0];
            const float sc = mw == kNegInf ? 0.f : fast_exp2(mw - M);
            L += sc * s_ml[w][g][1];
            O0 += sc * s_acc[w][g][d];
            O1 += sc * s_acc[w][g][d + 1];
        }
        const int head = kvh * G + g;
        if (n_parts == 1) {
            float* orow = reinterpret_cast<float*>(p.out) + (int64_t)seq * p.out_st + (int64_t)head * p.out_sh;
            orow[d] = O0 / L;
            orow[d + 1] = O1 / L;
        } else {
            const int64_t slot = ((int64_t)seq * p.num_heads + head) * p.max_parts + part;
            put_pair<FUSED>(p.ws_o + slot * D + d, O0, O1);
            if (d == 0) put_pair<FUSED>(p.ws_ml + slot * 2, M, L);
        }
    }
    if (!FUSED || n_parts == 1) return;

    // ------------------------------------------------------------ merge the partitions
    // By the last workgroup of the (sequence, KV head) to get here, which returns the counter
    // to zero for the next call. The stores above are all this wave's: s_waitcnt vmcnt(0) holds
    // it until each is acknowledged from the agent's coherence point, before the counter moves.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint32_t* cnt = p.ws_cnt + ((int64_t)seq * p.num_kv_heads + kvh);
    uint32_t arrived = 0;
    if (lane == 0) arrived = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(arrived) != (uint32_t)(n_parts - 1)) return;
    if (lane == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    merge_partitions<D, G, true>(p, seq, kvh, n_parts);
}

// The same merge as a launch of its own, one wave per (KV head, sequence).
template <int D, int G>
__global__ __launch_bounds__(64) void paged_decode_combine_kernel(const AttnParams p) {
    const int kvh = (int)blockIdx.x;
    const int seq = (int)blockIdx.y;
    int64_t ctx64 = p.ctx_lens[seq];
    ctx64 = ctx64 < (int64_t)p.table_width * kBS ? ctx64 : (int64_t)p.table_width * kBS;
    ctx64 = ctx64 < (int64_t)p.max_parts * kDecodePart ? ctx64 : (int64_t)p.max_parts * kDecodePart;
    const int n_parts = (int)((ctx64 + kDecodePart - 1) / kDecodePart);
    if (n_parts > 1) merge_partitions<D, G, false>(p, seq, kvh, n_parts);
}

// Workgroups, at the bound of the launch, up to which it appends and merges by itself. us a call
// against three launches (append, partitions, merge), with the append, 12 heads, eager and
// replayed: 2 sequences of 4-1107 tokens 18.1 -> 13.6, 10.1 -> 8.0; 8 of 16-500 18.5 -> 13.5, 10.9
// -> 8.4; 32 of 16-1024 25.4 -> 21.7, 24.8 -> 22.0. Above, the waves that stay for the merge cost
// more than the launches: 64 of 200-3000 replayed, 9216 workgroups, 108.9 -> 115.7; 200 of
// 500-2000 272 -> 280. Both forms compute the same bits, whichever a captured step's bound takes.
constexpr int64_t kFusedWgs = 2048;

bool fused_size(const AttnParams& p) { return (int64_t)p.num_seqs * p.num_kv_heads * p.max_parts <= kFusedWgs; }

template <int D, int G>
int launch_g(const AttnParams& p, dim3 grid, hipStream_t stream) {
    const bool fused = fused_size(p) && (p.max_parts == 1 ? p.app_slots != nullptr : p.ws_cnt != nullptr);
    if (fused) paged_decode_kernel<D, G, true><<<grid, kWaves * 64, 0, stream>>>(p);
    else paged_decode_kernel<D, G, false><<<grid, kWaves * 64, 0, stream>>>(p);
    int rc = check_launch("paged decode attention");
    if (rc || fused || p.max_parts == 1) return rc;
    paged_decode_combine_kernel<D, G><<<dim3(grid.x, grid.z), 64, 0, stream>>>(p);
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

bool decode_f32_appends(const AttnParams& p) {
    if (!fused_size(p) || (p.max_parts > 1 && !p.ws_cnt)) return false;
    return (((uint64_t)(uintptr_t)p.app_k | (uint64_t)(uintptr_t)p.app_v | (uint64_t)(p.app_st * 4) |
             (uint64_t)(p.app_sh * 4)) % 16) == 0;
}

int launch_decode_f32(const AttnParams& p, hipStream_t stream) {
    if (!decode_f32_applies(p)) return PKV_EUNSUPPORTED;
    const dim3 grid((unsigned)p.num_kv_heads, (unsigned)p.max_parts, (unsigned)p.num_seqs);
    return p.group == 1 ? launch_g<64, 1>(p, grid, stream) : launch_g<64, 2>(p, grid, stream);
}

}  // namespace pkv
