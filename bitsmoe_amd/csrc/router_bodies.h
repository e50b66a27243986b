// Device bodies of the router: top-k of a token by counting, and the router's linear layer with it.
#pragma once
#include "common.h"

namespace bitsmoe {

__device__ inline float wave_sum(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
    return v;
}

// The same result for at most 256 experts without the k dependent arg-max rounds: every lane
// counts, for each of its (up to four) logits, how many of the token's logits precede it in
// the order (value descending, expert index ascending); that count is the position of the
// expert in the top-k list.  The logits of a token sit in LDS and are read as broadcasts.
// grid = ceil(T / 4), 256 threads (one wavefront per token).
constexpr int ROUTER_RANK_PER_LANE = 4;
template <int NW>      // wavefronts per workgroup
struct RankTopkLds {
    // sort key of a logit: the float mapped to an unsigned integer of the same order, above the
    // complemented expert index, so that one 64-bit comparison is "precedes in the top-k order"
    uint64_t keys[NW][64 * ROUTER_RANK_PER_LANE];
    float picked[NW][64];
};
// One token by one wavefront (`wv` of its workgroup): v[i] is the logit of expert lane + 64 i (-inf past E).
// LIVE: logits per lane that can exist (E <= 64 LIVE); the counting loop, which is most of the work, runs over those only.
template <int LIVE, int NW>
__device__ inline void rank_topk_live(float (&v)[ROUTER_RANK_PER_LANE], RankTopkLds<NW>& lds, int wv, int lane, int tkn, float wscale,
                                      int E, int k, int renorm, int round_dt, int32_t* __restrict__ sel32,
                                      int64_t* __restrict__ sel64, float* __restrict__ weights) {
    const int e2 = (E + 1) & ~1;
    uint64_t mine[LIVE];
    float vmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < LIVE; ++i) {
        const int e = lane + 64 * i;
        vmax = fmaxf(vmax, v[i]);
        const uint32_t bits = __float_as_uint(v[i] + 0.0f);      // (-0 and +0 are one value)
        const uint32_t ordered = bits ^ ((bits >> 31) ? 0xFFFFFFFFu : 0x80000000u);
        mine[i] = e < E ? ((uint64_t)ordered << 32) | (uint32_t)(0xFFFFFFFFu - (uint32_t)e) : 0ull;   // padding sorts last
        lds.keys[wv][e] = mine[i];
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) vmax = fmaxf(vmax, __shfl_xor(vmax, d));
    float pr[LIVE];
    float part = 0.0f;
#pragma unroll
    for (int i = 0; i < LIVE; ++i) {
        pr[i] = (v[i] == -INFINITY) ? 0.0f : expf(v[i] - vmax);
        part += pr[i];
    }
    const float denom = wave_sum(part);
    // the other lanes' keys are read below: order the LDS writes above before those reads whatever
    // the compiler's schedule (one wavefront: a wave-scope fence and a wave barrier, no s_barrier)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    int rank[LIVE] = {};
#pragma unroll 4
    for (int o = 0; o < e2; o += 2) {
        const uint64_t q0 = lds.keys[wv][o], q1 = lds.keys[wv][o + 1];
#pragma unroll
        for (int i = 0; i < LIVE; ++i) rank[i] += (int)(q0 > mine[i]) + (int)(q1 > mine[i]);
    }
#pragma unroll
    for (int i = 0; i < LIVE; ++i)
        if (lane + 64 * i < E && rank[i] < k) lds.picked[wv][rank[i]] = pr[i] / denom;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float picked_sum = 0.0f;
    for (int j = 0; j < k; ++j) picked_sum += lds.picked[wv][j];
#pragma unroll
    for (int i = 0; i < LIVE; ++i) {
        if (lane + 64 * i < E && rank[i] < k) {
            float w = pr[i] / denom;
            if (renorm) w /= picked_sum;
            w *= wscale;
            if (round_dt == BITSMOE_DT_F16)
                w = __half2float(__float2half(w));
            else if (round_dt == BITSMOE_DT_BF16)
                w = __bfloat162float(__float2bfloat16(w));
            const int64_t o = (int64_t)tkn * k + rank[i];
            if (sel32) sel32[o] = lane + 64 * i;
            if (sel64) sel64[o] = lane + 64 * i;
            weights[o] = w;
        }
    }
    // (the next token of this wavefront overwrites keys / picked: its reads above are done first)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int NW>
__device__ inline void rank_topk_token(float (&v)[ROUTER_RANK_PER_LANE], RankTopkLds<NW>& lds, int wv, int lane, int tkn, float wscale,
                                       int E, int k, int renorm, int round_dt, int32_t* __restrict__ sel32,
                                       int64_t* __restrict__ sel64, float* __restrict__ weights) {
    if (E <= 64)
        rank_topk_live<1>(v, lds, wv, lane, tkn, wscale, E, k, renorm, round_dt, sel32, sel64, weights);
    else if (E <= 128)
        rank_topk_live<2>(v, lds, wv, lane, tkn, wscale, E, k, renorm, round_dt, sel32, sel64, weights);
    else
        rank_topk_live<ROUTER_RANK_PER_LANE>(v, lds, wv, lane, tkn, wscale, E, k, renorm, round_dt, sel32, sel64, weights);
}

// The router's linear layer and the top-k in ONE kernel, for gates that compute their logits in fp32 from 16-bit
// hidden states and a 16-bit weight (DeepSeek-V2's gate: bitsmoe/models/deepseekv2/configuration_deepseek.py:125-139
// names its form; the reference calls the model's own gate module, bitsmoe/models/deepseekv2/bitsmoe_block.py:74):
// the products of 16-bit values are exact in fp32, so MFMA sums in fp32 are the module's logits up to summation
// order.  A workgroup of NW wavefronts takes 16 tokens: wavefront w contracts over the w-th part of the hidden size
// for all experts (NB 16-expert blocks; sixteen wavefronts: all its operands of a 2048-wide layer are ONE batch of
// loads), the partial sums meet in LDS (a tree in a fixed order: the same logits whenever the inputs are the same), then
// the wavefronts rank the tokens, 16 / NW each.
// x [T, K] and weight [E, K] are read as MFMA operands straight from memory (16 bytes per lane).
// PREP: the weight in MFMA operand order ([16-expert block][k-step of 32][lane][8 values]: bitsmoe_prepare_linear_weight):
// a wavefront's load is 1 KB of consecutive memory.
// TOKENS: of the sixteen rows of an MFMA (a workgroup beside another kernel's takes fewer, one per wavefront).
template <int NB, int NW>
struct RouterLinearLds {
    static constexpr int LD = NB * 16 + 1;
    // DIRECT: every wavefront's partial sums fit the LDS side by side and the ranking wavefront adds them up itself (one
    // barrier); otherwise a tree over half as many slots (slot 0 ends as the total).  Both add in a fixed order.
    static constexpr bool DIRECT = NW * 16 * LD * 4 + sizeof(RankTopkLds<NW>) <= 160 * 1024;
    float part[(DIRECT ? NW : NW / 2) * 16 * LD];
    __attribute__((aligned(16))) RankTopkLds<NW> rank;
};
template <bool BF16, int NB, int NW, bool PREP, int TOKENS>
__device__ __forceinline__ void router_linear_body(const uint16_t* __restrict__ x, int64_t ld_x, const uint16_t* __restrict__ weight, int T, int K,
                                                   int E, int k, float wscale, int renorm, int round_dt, int32_t* __restrict__ sel32,
                                                   int64_t* __restrict__ sel64, float* __restrict__ weights, int t0,
                                                   RouterLinearLds<NB, NW>& lds) {
    // k-steps whose operands are requested together (four wavefronts beside another kernel's: every further group is one more trip; with
    // half as many the launch at 64 experts and 12 rows takes 13.8 us instead of 12.8, with 128 experts as long)
    constexpr int U = (NB <= 4 ? 4 : NB <= 8 ? 2 : 1) * (TOKENS == 4 ? 2 : 1);
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
    typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
    constexpr int LD = RouterLinearLds<NB, NW>::LD;
    constexpr bool DIRECT = RouterLinearLds<NB, NW>::DIRECT;
    float* part = lds.part;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int row = t0 + min(lane & 15, TOKENS - 1);
    const int kq = K / NW;                       // contraction range of this wavefront (a multiple of 32)
    const int kbase = wv * kq + (lane >> 4) * 8;
    f32x4 acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const uint16_t* __restrict__ xp = x + (int64_t)min(row, T - 1) * ld_x + kbase;
    for (int s0 = 0; s0 < kq; s0 += 32 * U) {
        u32x4 a[U], b[U][NB];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int ks = min(s0 + 32 * u, kq - 32);      // (a short last group repeats its final step: masked below)
            a[u] = *reinterpret_cast<const u32x4*>(xp + ks);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                if constexpr (PREP) {
                    const int blk = min(nb, (E - 1) >> 4);      // (blocks past the last expert repeat it: masked below)
                    b[u][nb] = *reinterpret_cast<const u32x4*>(weight + (((int64_t)blk * (K >> 5) + ((wv * kq + ks) >> 5)) * 64 + lane) * 8);
                } else {
                    const int e = min(nb * 16 + (lane & 15), E - 1);
                    b[u][nb] = *reinterpret_cast<const u32x4*>(weight + (int64_t)e * K + kbase + ks);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);      // (every request of the group is out before its first MFMA)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // (no branch between the steps: a step past the end contributes zeros)
            const bool live = s0 + 32 * u < kq;
#pragma unroll
            for (int c = 0; c < 4; ++c) a[u][c] = live ? a[u][c] : 0u;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                if constexpr (BF16)
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[u]), __builtin_bit_cast(bf16x8, b[u][nb]),
                                                                      acc[nb], 0, 0, 0);
                else
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[u]), __builtin_bit_cast(f16x8, b[u][nb]),
                                                                     acc[nb], 0, 0, 0);
            }
        }
    }
    // lane holds tokens 4 (lane / 16) + j, expert 16 nb + lane % 16
    auto slot_of = [&](int w, int nb, int j) -> float& { return part[(w * 16 + 4 * (lane >> 4) + j) * LD + nb * 16 + (lane & 15)]; };
    if constexpr (DIRECT) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int j = 0; j < 4; ++j) slot_of(wv, nb, j) = acc[nb][j];
    }
    for (int half = DIRECT ? 0 : NW / 2; half >= 1; half >>= 1) {      // wavefronts [half, 2 half) hand their sums to [0, half)
        if (wv >= half && wv < 2 * half) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int j = 0; j < 4; ++j) slot_of(wv - half, nb, j) = acc[nb][j];
        }
        __syncthreads();
        if (wv < half) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[nb][j] += slot_of(wv, nb, j);
        }
        __syncthreads();
    }
    if (!DIRECT && wv == 0) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int j = 0; j < 4; ++j) slot_of(0, nb, j) = acc[nb][j];
    }
    __syncthreads();
    constexpr int PER = TOKENS / NW > 0 ? TOKENS / NW : 1;
    for (int i = 0; i < PER; ++i) {
        const int tl = wv * PER + i, tkn = t0 + tl;
        if (tl >= TOKENS || tkn >= T) break;       // (wave-uniform; no workgroup barrier below)
        float v[ROUTER_RANK_PER_LANE];
#pragma unroll
        for (int q = 0; q < ROUTER_RANK_PER_LANE; ++q) {
            const int e = lane + 64 * q;
            float sum = -INFINITY;
            if (e < E && e < NB * 16) {
                sum = part[tl * LD + e];
                if constexpr (DIRECT) {
#pragma unroll
                    for (int w = 1; w < NW; ++w) sum += part[(w * 16 + tl) * LD + e];
                }
            }
            v[q] = sum;
        }
        rank_topk_token(v, lds.rank, wv, lane, tkn, wscale, E, k, renorm, round_dt, sel32, sel64, weights);
    }
}

}  // namespace bitsmoe
