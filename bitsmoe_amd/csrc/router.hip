// Router front end in one kernel: softmax over the expert logits in fp32, top-k, optional
// renormalisation of the k probabilities, optional round trip of the weights through a 16-bit
// type.  Replaces the chain of framework ops of the reference's Qwen blocks
// (bitsmoe/models/qwen3moe/bitsmoe_block.py:45-51, bitsmoe/models/qwen3next/bitsmoe_block.py:92-98):
//     p = softmax(logits.float());  w, idx = topk(p, k);  w /= w.sum();  w = w.to(act dtype)
// One wavefront per token; a lane holds the logits of experts lane, lane + 64, ...
#include "common.h"
#include "router_bodies.h"

#include <algorithm>

namespace bitsmoe {

constexpr int ROUTER_MAX_PER_LANE = 16;   // experts <= 1024

template <int DT>   // 0: fp16, 1: bf16, 2: fp32 logits
__device__ inline float load_logit(const void* __restrict__ base, int64_t idx) {
    if constexpr (DT == 2) {
        return reinterpret_cast<const float*>(base)[idx];
    } else if constexpr (DT == 1) {
        return __uint_as_float((uint32_t)reinterpret_cast<const uint16_t*>(base)[idx] << 16);
    } else {
        return __half2float(reinterpret_cast<const __half*>(base)[idx]);
    }
}

// The value N lanes away inside a row of sixteen, and reductions of a wavefront to a uniform value by it: a row's in four
// rotations, the four rows' through scalar registers (the LDS crossbar's permutes: six dependent round trips).
template <int N>
__device__ __forceinline__ int row_ror(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x120 + N, 0xF, 0xF, false);
}
template <class F>
__device__ __forceinline__ int wave_fold(int v, F&& f) {
    v = f(v, row_ror<8>(v));
    v = f(v, row_ror<4>(v));
    v = f(v, row_ror<2>(v));
    v = f(v, row_ror<1>(v));
    return f(f(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             f(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}
__device__ __forceinline__ float wave_max(float v) {
    return __int_as_float(wave_fold(__float_as_int(v), [](int a, int b) { return __float_as_int(fmaxf(__int_as_float(a), __int_as_float(b))); }));
}
__device__ __forceinline__ int wave_min(int v) {
    return wave_fold(v, [](int a, int b) { return min(a, b); });
}

// grid = ceil(T / 4), 256 threads (four tokens per workgroup); PER: logits a lane holds, E <= 64 * PER.
// Bound by the chain of the k arg-max rounds: a round is PER compares, two reductions by row rotations, PER compares to take
// the pick out; exponentials and divisions come once, behind the rounds.  (With permutes, both parts of the pair in every
// step, sixteen logits per lane whatever E, and an exponential and a division per round: 512 experts, top-10, 256 tokens
// 12.6 -> 5.6 us; 4096 tokens 16.7 -> 10.2.)
template <int DT, int PER>
__global__ __launch_bounds__(256) void k_router_softmax_topk(const void* __restrict__ logits, int64_t ld, float wscale,
                                                             int T, int E, int k,
                                                             int renorm, int round_dt, int32_t* __restrict__ sel32,
                                                             int64_t* __restrict__ sel64, float* __restrict__ weights) {
    const int lane = threadIdx.x & 63;
    const int tkn = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tkn >= T) return;
    float v[PER];
    float vmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = lane + 64 * i;
        v[i] = e < E ? load_logit<DT>(logits, (int64_t)tkn * ld + e) : -INFINITY;
        vmax = fmaxf(vmax, v[i]);
    }
    vmax = wave_max(vmax);
    float part = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) part += (v[i] == -INFINITY) ? 0.0f : expf(v[i] - vmax);
    const float denom = wave_sum(part);

    // k rounds of arg-max over what is left; ties go to the lower expert index
    float my_v = -INFINITY;      // lane j < k keeps the j-th pick
    int my_e = 0;
    for (int j = 0; j < k; ++j) {
        float best = -INFINITY;
        int best_e = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (v[i] > best) {      // ascending e inside a lane: strict > keeps the lower index (and a NaN is never picked)
                best = v[i];
                best_e = lane + 64 * i;
            }
        }
        const float top = wave_max(best);
        const int top_e = wave_min(best == top ? best_e : 0x7fffffff);
        // remove the pick from its owner
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (lane + 64 * i == top_e) v[i] = -INFINITY;
        if (lane == j) {
            my_v = top;
            my_e = top_e < E ? top_e : 0;
        }
    }
    const float my_w = my_v == -INFINITY ? 0.0f : expf(my_v - vmax) / denom;
    float picked_sum = 0.0f;
    for (int j = 0; j < k; ++j) picked_sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_w), j));
    if (lane < k) {
        float w = (renorm ? my_w / picked_sum : my_w) * wscale;
        if (round_dt == BITSMOE_DT_F16)
            w = __half2float(__float2half(w));
        else if (round_dt == BITSMOE_DT_BF16)
            w = __bfloat162float(__float2bfloat16(w));
        const int64_t o = (int64_t)tkn * k + lane;
        if (sel32) sel32[o] = my_e;
        if (sel64) sel64[o] = my_e;
        weights[o] = w;
    }
}

template <int DT>
__global__ __launch_bounds__(256) void k_router_rank_topk(const void* __restrict__ logits, int64_t ld, float wscale, int T,
                                                          int E, int k,
                                                          int renorm, int round_dt, int32_t* __restrict__ sel32,
                                                          int64_t* __restrict__ sel64, float* __restrict__ weights) {
    __shared__ __attribute__((aligned(16))) RankTopkLds<4> lds;
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    const int tkn = blockIdx.x * 4 + wv;
    if (tkn >= T) return;            // (no workgroup barrier below: a wavefront only reads what it wrote)
    float v[ROUTER_RANK_PER_LANE];
#pragma unroll
    for (int i = 0; i < ROUTER_RANK_PER_LANE; ++i) {
        const int e = lane + 64 * i;
        v[i] = e < E ? load_logit<DT>(logits, (int64_t)tkn * ld + e) : -INFINITY;
    }
    rank_topk_token(v, lds, wv, lane, tkn, wscale, E, k, renorm, round_dt, sel32, sel64, weights);
}

template <bool BF16, int NB, int NW, bool PREP>
__global__ __launch_bounds__(NW * 64) void k_router_linear_topk(const uint16_t* __restrict__ x, int64_t ld_x,
                                                                const uint16_t* __restrict__ weight, int T, int K, int E, int k,
                                                                float wscale, int renorm, int round_dt,
                                                                int32_t* __restrict__ sel32, int64_t* __restrict__ sel64,
                                                                float* __restrict__ weights) {
    __shared__ __attribute__((aligned(16))) RouterLinearLds<NB, NW> lds;
    router_linear_body<BF16, NB, NW, PREP, 16>(x, ld_x, weight, T, K, E, k, wscale, renorm, round_dt, sel32, sel64, weights, blockIdx.x * 16, lds);
}

}  // namespace bitsmoe

using namespace bitsmoe;

extern "C" int bitsmoe_router_softmax_topk_strided(const void* logits, int32_t logits_dtype, int64_t ld_logits, int64_t n_tokens,
                                                   int32_t n_experts, int32_t top_k, int32_t renormalize, float weight_scale,
                                                   int32_t round_dtype, void* selected, int32_t ids_are_i64, float* weights,
                                                   void* stream) {
    BITSMOE_REQUIRE(n_tokens >= 0 && n_tokens < ((int64_t)1 << 31), "token count out of range");
    BITSMOE_REQUIRE(n_experts >= 1 && n_experts <= 64 * ROUTER_MAX_PER_LANE, "n_experts must be in [1, %d]",
                    64 * ROUTER_MAX_PER_LANE);
    BITSMOE_REQUIRE(top_k >= 1 && top_k <= 64 && top_k <= n_experts, "top_k must be in [1, min(64, n_experts)]");
    BITSMOE_REQUIRE(logits_dtype >= 0 && logits_dtype <= 2, "logits_dtype must be 0 (fp16), 1 (bf16) or 2 (fp32)");
    BITSMOE_REQUIRE(round_dtype >= -1 && round_dtype <= 1, "round_dtype must be -1 (none), 0 (fp16) or 1 (bf16)");
    BITSMOE_REQUIRE(ld_logits >= n_experts, "ld_logits must be at least n_experts");
    if (n_tokens == 0) return BITSMOE_OK;
    BITSMOE_REQUIRE(logits && selected && weights, "null pointer");
    hipStream_t st = (hipStream_t)stream;
    int32_t* s32 = ids_are_i64 ? nullptr : (int32_t*)selected;
    int64_t* s64 = ids_are_i64 ? (int64_t*)selected : nullptr;
    const dim3 grid((unsigned)((n_tokens + 3) / 4));
    const bool by_rank = n_experts <= 64 * ROUTER_RANK_PER_LANE;
#define BITSMOE_ROUTER_LAUNCH(KERNEL)                                                                              \
    hipLaunchKernelGGL(KERNEL, grid, dim3(256), 0, st, logits, ld_logits, weight_scale, (int)n_tokens, n_experts, top_k, \
                       renormalize, round_dtype, s32, s64, weights)
#define BITSMOE_ROUTER_FORM(DT)                                                                                    \
    do {                                                                                                           \
        if (by_rank) BITSMOE_ROUTER_LAUNCH((k_router_rank_topk<DT>));                                              \
        else if (n_experts <= 512) BITSMOE_ROUTER_LAUNCH((k_router_softmax_topk<DT, 8>));                          \
        else BITSMOE_ROUTER_LAUNCH((k_router_softmax_topk<DT, ROUTER_MAX_PER_LANE>));                              \
    } while (0)
    if (logits_dtype == 0) BITSMOE_ROUTER_FORM(0);
    else if (logits_dtype == 1) BITSMOE_ROUTER_FORM(1);
    else BITSMOE_ROUTER_FORM(2);
#undef BITSMOE_ROUTER_FORM
#undef BITSMOE_ROUTER_LAUNCH
    BITSMOE_HIP_TRY(hipGetLastError());
    return BITSMOE_OK;
}

extern "C" int bitsmoe_router_softmax_topk(const void* logits, int32_t logits_dtype, int64_t n_tokens, int32_t n_experts,
                                           int32_t top_k, int32_t renormalize, int32_t round_dtype, void* selected,
                                           int32_t ids_are_i64, float* weights, void* stream) {
    return bitsmoe_router_softmax_topk_strided(logits, logits_dtype, n_experts, n_tokens, n_experts, top_k, renormalize, 1.0f,
                                               round_dtype, selected, ids_are_i64, weights, stream);
}

extern "C" int bitsmoe_router_linear_topk(const void* hidden, int32_t dtype, int64_t ld_hidden, const void* weight,
                                          int32_t weight_is_prepared, int64_t n_tokens, int32_t hidden_size, int32_t n_experts, int32_t top_k,
                                          int32_t renormalize, float weight_scale, int32_t round_dtype, void* selected,
                                          int32_t ids_are_i64, float* weights, void* stream) {
    BITSMOE_REQUIRE(n_tokens >= 0 && n_tokens < ((int64_t)1 << 31), "token count out of range");
    BITSMOE_REQUIRE(dtype == BITSMOE_DT_F16 || dtype == BITSMOE_DT_BF16, "dtype must be f16 (0) or bf16 (1)");
    BITSMOE_REQUIRE(n_experts >= 1 && n_experts <= 64 * ROUTER_RANK_PER_LANE, "n_experts must be in [1, %d]", 64 * ROUTER_RANK_PER_LANE);
    BITSMOE_REQUIRE(top_k >= 1 && top_k <= 64 && top_k <= n_experts, "top_k must be in [1, min(64, n_experts)]");
    BITSMOE_REQUIRE(hidden_size >= 128 && hidden_size % 128 == 0, "hidden_size must be a positive multiple of 128");
    // (option router_wide = 0: four wavefronts per workgroup whatever the hidden size; experiments)
    const bool wide_wg = hidden_size % 512 == 0 && options().router_wide != 0;      // sixteen wavefronts, a sixteenth of the contraction each
    BITSMOE_REQUIRE(ld_hidden >= hidden_size && ld_hidden % 8 == 0, "ld_hidden must be at least hidden_size and a multiple of 8");
    BITSMOE_REQUIRE(round_dtype >= -1 && round_dtype <= 1, "round_dtype must be -1 (none), 0 (fp16) or 1 (bf16)");
    if (n_tokens == 0) return BITSMOE_OK;
    BITSMOE_REQUIRE(hidden && weight && selected && weights, "null pointer");
    BITSMOE_REQUIRE((((uintptr_t)hidden | (uintptr_t)weight) & 15) == 0, "hidden and weight must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    int32_t* s32 = ids_are_i64 ? nullptr : (int32_t*)selected;
    int64_t* s64 = ids_are_i64 ? (int64_t*)selected : nullptr;
    const dim3 grid((unsigned)((n_tokens + 15) / 16));
    const bool bf16 = dtype == BITSMOE_DT_BF16;
#define BITSMOE_ROUTER_LINEAR_P(B, NB, NWIDE, PR)                                                                             \
    do {                                                                                                                     \
        if (wide_wg)                                                                                                         \
            hipLaunchKernelGGL((k_router_linear_topk<B, NB, NWIDE, PR>), grid, dim3(NWIDE * 64), 0, st,                      \
                               (const uint16_t*)hidden, ld_hidden, (const uint16_t*)weight, (int)n_tokens, hidden_size,      \
                               n_experts, top_k, weight_scale, renormalize, round_dtype, s32, s64, weights);                 \
        else                                                                                                                 \
            hipLaunchKernelGGL((k_router_linear_topk<B, NB, 4, PR>), grid, dim3(256), 0, st, (const uint16_t*)hidden,        \
                               ld_hidden, (const uint16_t*)weight, (int)n_tokens, hidden_size, n_experts, top_k,             \
                               weight_scale, renormalize, round_dtype, s32, s64, weights);                                   \
    } while (0)
#define BITSMOE_ROUTER_LINEAR(B, NB, NWIDE)                                                      \
    do {                                                                                         \
        if (weight_is_prepared) BITSMOE_ROUTER_LINEAR_P(B, NB, NWIDE, true);                     \
        else BITSMOE_ROUTER_LINEAR_P(B, NB, NWIDE, false);                                       \
    } while (0)
    // (more than 128 experts: eight wavefronts, the partial sums of sixteen would not fit the LDS)
    if (n_experts <= 64) {
        if (bf16) BITSMOE_ROUTER_LINEAR(true, 4, 16); else BITSMOE_ROUTER_LINEAR(false, 4, 16);
    } else if (n_experts <= 128) {
        if (bf16) BITSMOE_ROUTER_LINEAR(true, 8, 16); else BITSMOE_ROUTER_LINEAR(false, 8, 16);
    } else {
        if (bf16) BITSMOE_ROUTER_LINEAR(true, 16, 8); else BITSMOE_ROUTER_LINEAR(false, 16, 8);
    }
#undef BITSMOE_ROUTER_LINEAR
#undef BITSMOE_ROUTER_LINEAR_P
    BITSMOE_HIP_TRY(hipGetLastError());
    return BITSMOE_OK;
}

// ---- the block's closing elementwise pass ---------------------------------------------------------------------------
// One row of the operand of the block's output GEMM, in the activation dtype:
//     out[t, 0 .. R)        = rank_accum[t, :]                                   (fp32 -> 16 bit)
//     out[t, R .. R + I_sh) = silu(a[t, c]) * b[t, c] * (g ? sigmoid(g[t]) : 1)   (the always-on shared expert's z)
// so that the routed experts' output projection and the shared expert's down projection are ONE GEMM against
// the stacked [U_down | W_down_shared] (bitsmoe/models/base_block.py:414, bitsmoe/models/qwen3next/bitsmoe_block.py:144-147,
// bitsmoe/models/deepseekv2/bitsmoe_block.py:123-124 run them as separate modules and add).  Eight elements per thread.
template <bool BF16>
__global__ __launch_bounds__(256) void k_block_finish(const float* __restrict__ rank_accum, int64_t T, int R,
                                                      const uint16_t* __restrict__ a, const uint16_t* __restrict__ b,
                                                      int64_t ld_ab, int I_sh, const uint16_t* __restrict__ g, int64_t ld_g,
                                                      uint16_t* __restrict__ out, int64_t ld_out, int c_first) {
    const int per_row = (R + I_sh - c_first) >> 3;      // (columns from c_first on)
    const int64_t total = T * per_row;
    auto to_f32 = [](uint16_t v) {
        if constexpr (BF16) return __uint_as_float((uint32_t)v << 16);
        else return __half2float(__ushort_as_half(v));
    };
    auto to_16 = [](float v) -> uint16_t {
        if constexpr (BF16) return __builtin_bit_cast(uint16_t, (__bf16)v);
        else return __builtin_bit_cast(uint16_t, (_Float16)v);
    };
    typedef uint32_t v4 __attribute__((ext_vector_type(4)));
    typedef float f4 __attribute__((ext_vector_type(4)));
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t t = i / per_row;
        const int c = c_first + (int)(i - t * per_row) * 8;
        uint16_t o[8];
        if (c < R) {
            const f4 lo = *reinterpret_cast<const f4*>(rank_accum + t * R + c);
            const f4 hi = *reinterpret_cast<const f4*>(rank_accum + t * R + c + 4);
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                o[x] = to_16(lo[x]);
                o[4 + x] = to_16(hi[x]);
            }
        } else {
            const int cs = c - R;
            const v4 av = *reinterpret_cast<const v4*>(a + t * ld_ab + cs);
            const v4 bv = *reinterpret_cast<const v4*>(b + t * ld_ab + cs);
            float gate = 1.0f;
            if (g) gate = 1.0f / (1.0f + __expf(-to_f32(g[t * ld_g])));
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const float a0 = to_f32((uint16_t)(av[x] & 0xFFFFu)), a1 = to_f32((uint16_t)(av[x] >> 16));
                const float b0 = to_f32((uint16_t)(bv[x] & 0xFFFFu)), b1 = to_f32((uint16_t)(bv[x] >> 16));
                // (rounded as the modules round: silu in the activation dtype, the product, the gate's scaling)
                o[2 * x] = to_16(to_f32(to_16(to_f32(to_16(a0 / (1.0f + __expf(-a0)))) * b0)) * gate);
                o[2 * x + 1] = to_16(to_f32(to_16(to_f32(to_16(a1 / (1.0f + __expf(-a1)))) * b1)) * gate);
            }
        }
        v4 packed;
#pragma unroll
        for (int x = 0; x < 4; ++x) packed[x] = (uint32_t)o[2 * x] | ((uint32_t)o[2 * x + 1] << 16);
        *reinterpret_cast<v4*>(out + t * ld_out + c) = packed;
    }
}

extern "C" int bitsmoe_block_finish(const float* rank_accum, int64_t n_tokens, int32_t rank_out, const void* shared_gate_out,
                                    const void* shared_up_out, int64_t ld_shared, int32_t shared_intermediate,
                                    const void* shared_gate_logit, int64_t ld_gate_logit, int32_t act_dtype, void* out,
                                    int64_t ld_out, void* stream) {
    return bitsmoe::block_finish(rank_accum, n_tokens, rank_out, shared_gate_out, shared_up_out, ld_shared, shared_intermediate,
                                 shared_gate_logit, ld_gate_logit, act_dtype, out, ld_out, false, stream);
}

int bitsmoe::block_finish(const float* rank_accum, int64_t n_tokens, int32_t rank_out, const void* shared_gate_out,
                          const void* shared_up_out, int64_t ld_shared, int32_t shared_intermediate, const void* shared_gate_logit,
                          int64_t ld_gate_logit, int32_t act_dtype, void* out, int64_t ld_out, bool shared_only, void* stream) {
    BITSMOE_REQUIRE(n_tokens >= 0 && rank_out > 0 && shared_intermediate >= 0, "negative size");
    BITSMOE_REQUIRE(rank_out % 8 == 0 && shared_intermediate % 8 == 0, "rank_out and shared_intermediate must be multiples of 8");
    BITSMOE_REQUIRE(act_dtype == BITSMOE_DT_F16 || act_dtype == BITSMOE_DT_BF16, "act_dtype must be f16 (0) or bf16 (1)");
    BITSMOE_REQUIRE(ld_out >= rank_out + shared_intermediate && ld_out % 8 == 0, "ld_out too small or not a multiple of 8");
    if (n_tokens == 0) return BITSMOE_OK;
    BITSMOE_REQUIRE(rank_accum && out, "null pointer");
    BITSMOE_REQUIRE(((uintptr_t)rank_accum & 15) == 0 && ((uintptr_t)out & 15) == 0, "rank_accum and out must be 16-byte aligned");
    if (shared_intermediate > 0) {
        BITSMOE_REQUIRE(shared_gate_out && shared_up_out && ld_shared >= shared_intermediate && ld_shared % 8 == 0,
                        "shared expert operands missing, or their row stride is not a multiple of 8");
        BITSMOE_REQUIRE(((uintptr_t)shared_gate_out & 15) == 0 && ((uintptr_t)shared_up_out & 15) == 0,
                        "shared expert operands must be 16-byte aligned");
    }
    hipStream_t st = (hipStream_t)stream;
    const int c_first = shared_only ? rank_out : 0;
    const int64_t total = n_tokens * ((rank_out + shared_intermediate - c_first) / 8);
    if (total == 0) return BITSMOE_OK;
    const unsigned blocks = (unsigned)std::min<int64_t>((total + 255) / 256, 4096);
    if (act_dtype == BITSMOE_DT_BF16)
        hipLaunchKernelGGL(k_block_finish<true>, dim3(blocks), dim3(256), 0, st, rank_accum, n_tokens, rank_out,
                           (const uint16_t*)shared_gate_out, (const uint16_t*)shared_up_out, ld_shared, shared_intermediate,
                           (const uint16_t*)shared_gate_logit, ld_gate_logit, (uint16_t*)out, ld_out, c_first);
    else
        hipLaunchKernelGGL(k_block_finish<false>, dim3(blocks), dim3(256), 0, st, rank_accum, n_tokens, rank_out,
                           (const uint16_t*)shared_gate_out, (const uint16_t*)shared_up_out, ld_shared, shared_intermediate,
                           (const uint16_t*)shared_gate_logit, ld_gate_logit, (uint16_t*)out, ld_out, c_first);
    BITSMOE_HIP_TRY(hipGetLastError());
    return BITSMOE_OK;
}
