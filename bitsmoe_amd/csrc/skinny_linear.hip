// A bias-free linear layer for a FEW rows: out[T, N] = x[T, K] * W[N, K]^T with T <= 64, 16-bit x / W / out, fp32 sums.
// The two GEMMs around the routed-expert operator (the row-stacked shared-basis / router / shared-expert projections
// in, the column-stacked output projections out: bitsmoe/models/qwen3moe/bitsmoe_block.py:63-64,
// bitsmoe/models/base_block.py:414) are this shape at decode sizes: tens of MB of weights against a handful of tokens,
// i.e. a stream of W at HBM speed, which general GEMM kernels tiled for square problems reach a fraction of.
// W stays in the framework's [out_features, in_features] layout: a lane's 16 bytes of a weight row are eight
// consecutive contraction indices, which is what the 16x16x32 MFMA takes as its second operand.
// A workgroup owns 16 output columns; each of its wavefronts contracts a share of K and they add up in LDS.
//
// What bounds it: one trip to memory for W, and x, which EVERY workgroup reads in full (T / 16 bytes of x per byte of W,
// from L2).  So (a) a wavefront requests its whole share of W -- up to MAXS steps, 1 KB each -- before it multiplies anything:
// with batches of four steps the trips followed each other; (b) x is fetched in pieces of whole cache lines (a wavefront
// reads G * 64 consecutive bytes of a row, several rows per instruction), turned in LDS and read from there as operands:
// fetched in operand order a load touched 64 bytes of sixteen rows, and the launch grew by 4 us per sixteen rows.
// Longer contractions take eight wavefronts, so that a share stays within MAXS steps (beyond that: several passes).
// Prepared weights, graph of launches over 600 MB of weights, us per launch (the library GEMM on the same card; before, with
// batches of four steps and x in operand order, on another) at 1, 16, 32, 48, 64 rows:
//   2048 -> 4224 features: 6.4 (12.0;  6.1),  7.4 (11.9;  8.3),  9.0 (11.9; 12.1), 10.3 (12.3; 16.0), 12.4 (12.5; 19.4)
//   2048 -> 2048 features: 4.4 (11.0;  4.5),  4.7 (11.0;  5.4),  5.7 (11.2;  7.4),  6.3 (11.1;  9.6),  7.4 (11.6; 11.5)
//   4864 -> 2048 features: 7.9 (17.4;  7.7),  8.2 (17.4;  9.8), 10.3 (13.8; 14.1), 13.4 (13.9; 19.7), 15.8 (16.3; 24.6)
//   2048 -> 9728 features: 9.7 (15.9;  9.9), 11.1 (14.4; 12.6), 13.0 (14.4; 18.1), 15.2 (15.5; 23.5), 17.6 (15.5; 28.6)
// (Shares that are no whole passes -- 4864 features are eight of nineteen steps -- pay for their selects: 0.5 to 1 us.)
#include "common.h"
#include "router_bodies.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace bitsmoe {

typedef float sk_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t sk_u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 sk_f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 sk_bf16x8 __attribute__((ext_vector_type(8)));

// XF32: x is fp32 and is rounded to the 16-bit type on its way into the MFMA (the cast of the operator's fp32 output in
// front of the output projection, bitsmoe/models/base_block.py:414, without a pass of its own).
// PREP: W was re-laid out once (bitsmoe_prepare_linear_weight) into the order the MFMA takes it: [16-column block]
// [k-step of 32][lane][8 values], so that a wavefront's load is 1 KB of consecutive memory instead of sixteen 64-byte
// pieces of sixteen rows.
// TURN: x by way of LDS; else (a few rows: nothing to gain from whole lines) every step's operand straight from x.
template <int NMB, int NW, bool XF32, bool TURN>
constexpr int SKINNY_LDS_BYTES = std::max(TURN ? NW * 16 * NMB * 32 * (NMB <= (XF32 ? 1 : 2) ? 4 : 2) * (XF32 ? 4 : 2) : 0, NW * NMB * 16 * 17 * 4);

template <bool BF16, int NMB, int NW, int MAXS, bool XF32, bool PREP, bool TURN, bool WHOLE>
__device__ __forceinline__ void skinny_body(const void* __restrict__ x, int64_t ld_x, const uint16_t* __restrict__ w, int T, int K, int N,
                                            uint16_t* __restrict__ out, int64_t ld_out, const float* __restrict__ addend, int64_t ld_add,
                                            int column_block, unsigned char* lds, unsigned char* zero_piece) {
    static_assert(TURN || NMB == 1, "few rows: one block of 16 rows");
    constexpr int G = NMB <= (XF32 ? 1 : 2) ? 4 : 2;   // k-steps per piece of x
    static_assert(MAXS % G == 0, "whole pieces");
    constexpr int EB = XF32 ? 4 : 2;                   // bytes of an element of x
    constexpr int CPR = 32 * G * EB / 16;              // 16-byte chunks per row of a piece
    constexpr int RPI = 64 / CPR;                      // rows per load instruction
    constexpr int NI = 16 * NMB / RPI;                 // load instructions per piece
    constexpr int PIECE = TURN ? 16 * NMB * CPR * 16 : 0;      // bytes
    constexpr int PART = NW * NMB * 16 * 17 * 4;
    static_assert((NW * PIECE > PART ? NW * PIECE : PART) == SKINNY_LDS_BYTES<NMB, NW, XF32, TURN>, "the kernel's LDS");
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, kg = lane >> 4;
    const int n0 = column_block * 16;
    if (TURN && lane == 0) *reinterpret_cast<sk_u32x4*>(zero_piece) = sk_u32x4{0u, 0u, 0u, 0u};      // (by every wavefront: no barrier)
    const int steps = K >> 5;
    const int first = wv * steps / NW, end = (wv + 1) * steps / NW;
    // chunk c of row r sits at chunk position c ^ swz(r) of its row: the sixteen rows of an operand read hit different banks
    auto swz = [](int r) { return CPR == 8 ? (r >> 1) & 7 : r & 15; };
    unsigned char* piece = lds + wv * PIECE;
    const unsigned char* xrow[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int r = i * RPI + lane / CPR;
        xrow[i] = (const unsigned char*)x + (int64_t)min(r, T - 1) * ld_x * EB + ((lane % CPR) ^ swz(r)) * 16;
    }
    const uint16_t* wp = PREP ? w + ((int64_t)column_block * steps) * 512 + lane * 8 : w + (int64_t)min(n0 + n, N - 1) * K + kg * 8;
    sk_f32x4 acc[NMB];
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) acc[mb] = sk_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto round16 = [](float v) -> uint32_t {
        if constexpr (BF16)
            return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)v);
        else
            return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v);
    };
    auto multiply = [&](sk_f32x4& c, sk_u32x4 av, sk_u32x4 bv) {
        if constexpr (BF16)
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sk_bf16x8, av), __builtin_bit_cast(sk_bf16x8, bv), c, 0, 0, 0);
        else
            c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(sk_f16x8, av), __builtin_bit_cast(sk_f16x8, bv), c, 0, 0, 0);
    };
    auto rounded = [&](sk_f32x4 lo, sk_f32x4 hi) {
        return sk_u32x4{round16(lo[0]) | (round16(lo[1]) << 16), round16(lo[2]) | (round16(lo[3]) << 16),
                        round16(hi[0]) | (round16(hi[1]) << 16), round16(hi[2]) | (round16(hi[3]) << 16)};
    };
    for (int s0 = first; s0 < end; s0 += MAXS) {
        // (no branches between the steps: those past the end repeat the last one and count as zeros -- both operands, or an
        // infinite x would make a NaN of its row; from LDS, x comes from a zero piece there: one select per operand, not four.
        // WHOLE: every share is whole passes of MAXS steps, no selects: with four per operand and step they were 0.3 to 1 us of a
        // launch.  A choice between the two bodies inside the kernel cost 1 to 3 us at 64 rows, in registers.)
        const int ns = end - s0;
        sk_u32x4 b[MAXS];
        auto request_w = [&](int u) {
            b[u] = *reinterpret_cast<const sk_u32x4*>(wp + (int64_t)(s0 + min(u, ns - 1)) * (PREP ? 512 : 32));
        };
        auto live_or_zero = [&](int u, sk_u32x4 v) {
            if constexpr (!WHOLE) {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = u < ns ? v[i] : 0u;
            }
            return v;
        };
        if constexpr (!TURN) {
            sk_u32x4 xr[MAXS][XF32 ? 2 : 1];
            const unsigned char* row = (const unsigned char*)x + ((int64_t)min(n, T - 1) * ld_x + kg * 8) * EB;
#pragma unroll
            for (int u = 0; u < MAXS; ++u) {
#pragma unroll
                for (int q = 0; q < (XF32 ? 2 : 1); ++q)
                    xr[u][q] = *reinterpret_cast<const sk_u32x4*>(row + (int64_t)(s0 + min(u, ns - 1)) * (32 * EB) + 16 * q);
                request_w(u);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < MAXS; ++u) {
                sk_u32x4 av = xr[u][0];
                if constexpr (XF32) av = rounded(__builtin_bit_cast(sk_f32x4, xr[u][0]), __builtin_bit_cast(sk_f32x4, xr[u][1]));
                multiply(acc[0], live_or_zero(u, av), live_or_zero(u, b[u]));
            }
            continue;
        }
        sk_u32x4 xr[2][NI];
        auto request_x = [&](auto p_c) {
            constexpr int P = decltype(p_c)::value;
            // (a piece that would stick out of the row is moved back: its steps are found `shift` further up)
            const int at = min(s0 + P * G, steps - G);
#pragma unroll
            for (int i = 0; i < NI; ++i) xr[P & 1][i] = *reinterpret_cast<const sk_u32x4*>(xrow[i] + (int64_t)at * (32 * EB));
        };
        // (x first: loads return in the order they are asked for, and x is the one that comes from L2)
        request_x(std::integral_constant<int, 0>{});
        if constexpr (MAXS > G) request_x(std::integral_constant<int, 1>{});
#pragma unroll
        for (int u = 0; u < MAXS; ++u) request_w(u);
        __builtin_amdgcn_sched_barrier(0);
        static_for([&](auto p_c) {
            constexpr int P = decltype(p_c)::value;
#pragma unroll
            for (int i = 0; i < NI; ++i) *reinterpret_cast<sk_u32x4*>(piece + (i * 64 + lane) * 16) = xr[P & 1][i];
            if constexpr ((P + 2) * G < MAXS) request_x(std::integral_constant<int, P + 2>{});
            __builtin_amdgcn_sched_barrier(0);
            const int shift = WHOLE ? 0 : s0 + P * G - min(s0 + P * G, steps - G);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const sk_u32x4 bv = live_or_zero(P * G + g, b[P * G + g]);
                const int gs = min(g + shift, G - 1);
                auto chunk = [&](int r, int c) -> const unsigned char* {
                    const unsigned char* at = piece + r * (CPR * 16) + ((c ^ swz(r)) << 4);
                    return WHOLE || P * G + g < ns ? at : zero_piece;
                };
#pragma unroll
                for (int mb = 0; mb < NMB; ++mb) {
                    const int r = 16 * mb + n;
                    if constexpr (XF32)
                        multiply(acc[mb], rounded(*reinterpret_cast<const sk_f32x4*>(chunk(r, gs * 8 + 2 * kg)),
                                                  *reinterpret_cast<const sk_f32x4*>(chunk(r, gs * 8 + 2 * kg + 1))), bv);
                    else
                        multiply(acc[mb], *reinterpret_cast<const sk_u32x4*>(chunk(r, gs * 4 + kg)), bv);
                }
            }
        }, std::make_integer_sequence<int, MAXS / G>{});
    }
    // lane holds rows 16 mb + 4 kg + j, column n; the partial sums take the place of the pieces of x
    auto part = [&](int w_, int row, int col) -> float& { return reinterpret_cast<float*>(lds)[(w_ * (NMB * 16) + row) * 17 + col]; };
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
        for (int j = 0; j < 4; ++j) part(wv, mb * 16 + 4 * kg + j, n) = acc[mb][j];
    __syncthreads();
    // the partial sums in a fixed order, two neighbouring columns per thread
    for (int i = threadIdx.x; i < NMB * 16 * 8; i += 64 * NW) {
        const int row = i / 8, c = (i % 8) * 2;
        if (row >= T || n0 + c >= N) continue;
        float v0 = 0.0f, v1 = 0.0f;
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            v0 += part(q, row, c);
            v1 += part(q, row, c + 1);
        }
        if (addend) {      // (fp32 [T, N] added to the sums before the one rounding of the result)
            v0 += addend[(int64_t)row * ld_add + n0 + c];
            v1 += addend[(int64_t)row * ld_add + n0 + c + 1];
        }
        *reinterpret_cast<uint32_t*>(out + (int64_t)row * ld_out + n0 + c) = round16(v0) | (round16(v1) << 16);
    }
}

template <bool BF16, int NMB, int NW, int MAXS, bool XF32, bool PREP, bool TURN, bool WHOLE>
__global__ __launch_bounds__(64 * NW) void k_skinny_linear(const void* __restrict__ x, int64_t ld_x, const uint16_t* __restrict__ w,
                                                           int T, int K, int N, uint16_t* __restrict__ out, int64_t ld_out,
                                                           const float* __restrict__ addend, int64_t ld_add) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[SKINNY_LDS_BYTES<NMB, NW, XF32, TURN>];
    __shared__ __attribute__((aligned(16))) unsigned char zero_piece[16];
    skinny_body<BF16, NMB, NW, MAXS, XF32, PREP, TURN, WHOLE>(x, ld_x, w, T, K, N, out, ld_out, addend, ld_add, blockIdx.x, lds, zero_piece);
}

// The input projection and, in its first `router_blocks` workgroups, the router's linear layer and top-k of four tokens each: both read
// the hidden states only.  What bounds the router is what one CU can fetch (256 KB of gate weight at 64 experts and a hidden size of 2048), so
// on its own it takes about as long as the projection, on a card that is idle but for one workgroup per sixteen tokens; here
// it is over before the projection is.  us, projection + router -> joint, 64 experts: 12 rows 11.1 + 10.2 -> 12.8; blocks in a graph at 1, 12 and
// 40 tokens 36.6 -> 32.1, 72.8 -> 63.7, 91.7 -> 79.9; 128 experts at 12 and 40 tokens 70.9 -> 61.4, 105.4 -> 88.5.  Blocks of 8 to 128
// experts, hidden sizes 1024 to 2560, 1 to 48 tokens: 0.85 of the time on average, none of 385 slower.  Contractions that are no
// four whole shares (3072, 4096, 5120) and more than 128 experts have no joint form built: they run the two launches.
template <bool BF16, int NMB, int MAXS, bool TURN, int NB>      // NB: 16-expert blocks
__global__ __launch_bounds__(256) void k_skinny_linear_router(const void* __restrict__ x, int64_t ld_x, const uint16_t* __restrict__ w, int T,
                                                              int K, int N, uint16_t* __restrict__ out, int64_t ld_out, int router_blocks,
                                                              const RouterBeside r) {
    using RouterLds = RouterLinearLds<NB, 4>;
    constexpr int BYTES = std::max((int)sizeof(RouterLds), SKINNY_LDS_BYTES<NMB, 4, false, TURN>);
    __shared__ __attribute__((aligned(16))) unsigned char lds[BYTES];
    __shared__ __attribute__((aligned(16))) unsigned char zero_piece[16];
    if ((int)blockIdx.x < router_blocks)
        router_linear_body<BF16, NB, 4, true, 4>((const uint16_t*)x, ld_x, (const uint16_t*)r.weight, T, K, r.n_experts, r.top_k,
                                                               r.weight_scale, r.renormalize, r.round_dtype, nullptr, r.selected, r.weights,
                                                               blockIdx.x * 4, *reinterpret_cast<RouterLds*>(lds));
    else
        skinny_body<BF16, NMB, 4, MAXS, false, true, TURN, true>(x, ld_x, w, T, K, N, out, ld_out, nullptr, 0, blockIdx.x - router_blocks, lds,
                                                                 zero_piece);
}

// W [N, K] -> [ceil(N / 16)][K / 32][64 lanes][8]: lane = 16 * (k % 32 / 8) + n % 16 holds W[n][32 ks + 8 (lane / 16) .. + 7];
// rows past N are zeros.  One thread per 16-byte piece.
__global__ __launch_bounds__(256) void k_prepare_linear_weight(const uint16_t* __restrict__ w, int N, int K, uint16_t* __restrict__ out,
                                                               int64_t pieces) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= pieces) return;
    const int lane = (int)(i & 63);
    const int64_t blk = i >> 6;
    const int ksteps = K >> 5;
    const int ks = (int)(blk % ksteps), nb = (int)(blk / ksteps);
    const int n = nb * 16 + (lane & 15), k = ks * 32 + (lane >> 4) * 8;
    sk_u32x4 v = {0u, 0u, 0u, 0u};
    if (n < N) v = *reinterpret_cast<const sk_u32x4*>(w + (int64_t)n * K + k);
    *reinterpret_cast<sk_u32x4*>(out + i * 8) = v;
}

}  // namespace bitsmoe

using namespace bitsmoe;

extern "C" int64_t bitsmoe_prepared_linear_weight_elements(int32_t in_features, int32_t out_features) {
    if (in_features <= 0 || out_features <= 0) return 0;
    return (int64_t)((out_features + 15) / 16) * 16 * in_features;
}

extern "C" int bitsmoe_prepare_linear_weight(const void* weight, int32_t in_features, int32_t out_features, void* prepared,
                                             void* stream) {
    BITSMOE_REQUIRE(in_features >= 128 && in_features % 128 == 0, "in_features must be a positive multiple of 128");
    BITSMOE_REQUIRE(out_features >= 1, "out_features must be positive");
    BITSMOE_REQUIRE(weight && prepared, "null pointer");
    BITSMOE_REQUIRE((((uintptr_t)weight | (uintptr_t)prepared) & 15) == 0, "weight and prepared must be 16-byte aligned");
    const int64_t pieces = bitsmoe_prepared_linear_weight_elements(in_features, out_features) / 8;
    hipLaunchKernelGGL(k_prepare_linear_weight, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t*)weight, out_features, in_features, (uint16_t*)prepared, pieces);
    BITSMOE_HIP_TRY(hipGetLastError());
    return BITSMOE_OK;
}

extern "C" int bitsmoe_skinny_linear(const void* x, int32_t dtype, int32_t x_is_f32, int64_t ld_x, const void* weight,
                                     int32_t weight_is_prepared, int64_t n_rows, int32_t in_features, int32_t out_features,
                                     void* out, int64_t ld_out, const float* addend, int64_t ld_addend, void* stream) {
    BITSMOE_REQUIRE(!x_is_f32 || n_rows <= 16, "n_rows must be in [0, 64] (fp32 rows: [0, 16])");
    return bitsmoe::skinny_linear(x, dtype, x_is_f32, ld_x, weight, weight_is_prepared, n_rows, in_features, out_features, out, ld_out,
                                  addend, ld_addend, stream);
}

// Up to sixteen rows always; seventeen to 32 with prepared weights of up to 1536 features (shares of up to twelve steps).  Instead of a
// pass that rounds them, every workgroup fetches twice the bytes of x, which shows from 2048 features on.  Graph of four layers of a
// block, us per layer, pass -> fp32 rows, at 17, 20, 26 and 32 tokens (runs of one side differ by 0.3 us):
//   1024 features:  34.2 -> 33.3  34.3 -> 33.4  45.1 -> 44.4  46.5 -> 45.7
//   1536 features:  42.4 -> 41.7  43.3 -> 42.4  44.0 -> 43.1  42.6 -> 41.9
//   2048 features, 32 experts:  51.1 -> 50.8  53.5 -> 53.2  53.9 -> 53.6  56.0 -> 55.5
//   2048 features, 128 experts:  67.1 -> 66.9  68.4 -> 68.3  (32 tokens) 72.5 -> 72.5  (48) 78.2 -> 79.8  (64) 83.1 -> 85.9
//   2560 features:  70.0 -> 70.7  72.2 -> 72.7  74.9 -> 75.6  73.7 -> 74.6
bool bitsmoe::skinny_f32_rows_possible(int64_t n_rows, int32_t in_features, int32_t weight_is_prepared) {
    return n_rows <= 16 || (n_rows <= 32 && weight_is_prepared != 0 && in_features <= 48 * 32);
}

int bitsmoe::skinny_linear(const void* x, int32_t dtype, int32_t x_is_f32, int64_t ld_x, const void* weight, int32_t weight_is_prepared,
                           int64_t n_rows, int32_t in_features, int32_t out_features, void* out, int64_t ld_out, const float* addend,
                           int64_t ld_addend, void* stream) {
    BITSMOE_REQUIRE(dtype == BITSMOE_DT_F16 || dtype == BITSMOE_DT_BF16, "dtype must be f16 (0) or bf16 (1)");
    BITSMOE_REQUIRE(n_rows >= 0 && n_rows <= 64, "n_rows must be in [0, 64] (fp32 rows: [0, 16])");
    BITSMOE_REQUIRE(!x_is_f32 || skinny_f32_rows_possible(n_rows, in_features, weight_is_prepared),
                    "more than 16 fp32 rows: at most 32, and prepared weights of at most 1536 features");
    BITSMOE_REQUIRE(in_features >= 128 && in_features % 128 == 0, "in_features must be a positive multiple of 128");
    BITSMOE_REQUIRE(out_features >= 2 && out_features % 2 == 0, "out_features must be even");
    BITSMOE_REQUIRE(ld_x >= in_features && ld_x % (x_is_f32 ? 4 : 8) == 0,
                    "ld_x must be at least in_features and a multiple of 8 (fp32 rows: of 4)");
    BITSMOE_REQUIRE(ld_out >= out_features && ld_out % 2 == 0, "ld_out must be at least out_features and even");
    BITSMOE_REQUIRE(addend == nullptr || ld_addend >= out_features, "ld_addend must be at least out_features");
    if (n_rows == 0) return BITSMOE_OK;
    BITSMOE_REQUIRE(x && weight && out, "null pointer");
    BITSMOE_REQUIRE((((uintptr_t)x | (uintptr_t)weight) & 15) == 0 && ((uintptr_t)out & 3) == 0,
                    "x and weight must be 16-byte aligned, out 4-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    const int nmb = (int)((n_rows + 15) / 16);
    const dim3 grid((unsigned)((out_features + 15) / 16));
    // a wavefront's share of the contraction, with four wavefronts or (shares of more than twenty steps) eight
    const int steps = in_features / 32;
    const int nw = steps > 80 ? 8 : 4;
    const int share = (steps + nw - 1) / nw;
    auto run = [&](auto bf_c, auto nmb_c, auto nw_c, auto s_c, auto xf_c, auto pr_c, auto turn_c) {
        auto launch = [&](auto whole_c) {
            hipLaunchKernelGGL((k_skinny_linear<decltype(bf_c)::value, decltype(nmb_c)::value, decltype(nw_c)::value, decltype(s_c)::value,
                                                decltype(xf_c)::value, decltype(pr_c)::value, decltype(turn_c)::value, decltype(whole_c)::value>),
                               grid, dim3(64 * decltype(nw_c)::value), 0, st, x, ld_x, (const uint16_t*)weight, (int)n_rows, in_features,
                               out_features, (uint16_t*)out, ld_out, addend, ld_addend);
        };
        // (hidden sizes 1024, 1536, 2048 and 2560 are four whole shares of prepared weights)
        if constexpr (decltype(pr_c)::value && decltype(nw_c)::value == 4) {
            if (steps % (4 * decltype(s_c)::value) == 0) return launch(std::true_type{});
        }
        launch(std::false_type{});
    };
    using std::integral_constant;
    using Yes = std::true_type;
    using No = std::false_type;
    using W4 = integral_constant<int, 4>;
    using W8 = integral_constant<int, 8>;
    using S8 = integral_constant<int, 8>;
    using S12 = integral_constant<int, 12>;
    using S16 = integral_constant<int, 16>;
    using S20 = integral_constant<int, 20>;
    auto by_share = [&](auto bf_c, auto nmb_c, auto xf_c, auto turn_c) {
        constexpr bool twenty = !(decltype(xf_c)::value && !decltype(turn_c)::value);      // (fp32 operands of twenty steps do not fit the registers)
        constexpr bool many_f32 = decltype(xf_c)::value && decltype(nmb_c)::value > 1;
        if constexpr (many_f32) {       // (prepared, four wavefronts, up to twelve steps: skinny_f32_rows_possible)
            if (share <= 8) run(bf_c, nmb_c, W4{}, S8{}, xf_c, Yes{}, turn_c);
            else run(bf_c, nmb_c, W4{}, S12{}, xf_c, Yes{}, turn_c);
        } else if (!weight_is_prepared) {      // (in passes of sixteen steps: the same sums in the same order)
            if (nw == 8) run(bf_c, nmb_c, W8{}, S16{}, xf_c, No{}, turn_c); else run(bf_c, nmb_c, W4{}, S16{}, xf_c, No{}, turn_c);
        } else if (nw == 8) {
            if (share <= 16 || !twenty) run(bf_c, nmb_c, W8{}, S16{}, xf_c, Yes{}, turn_c);
            else if constexpr (twenty) run(bf_c, nmb_c, W8{}, S20{}, xf_c, Yes{}, turn_c);
        } else if (share <= 8) {
            run(bf_c, nmb_c, W4{}, S8{}, xf_c, Yes{}, turn_c);
        } else if (share <= 12) {      // (1536 -> 4224 features at one row 6.0 us as sixteen steps, 5.6 as twelve)
            run(bf_c, nmb_c, W4{}, S12{}, xf_c, Yes{}, turn_c);
        } else {
            if (share <= 16 || !twenty) run(bf_c, nmb_c, W4{}, S16{}, xf_c, Yes{}, turn_c);
            else if constexpr (twenty) run(bf_c, nmb_c, W4{}, S20{}, xf_c, Yes{}, turn_c);
        }
    };
    auto by_rows = [&](auto bf_c) {
        using One = integral_constant<int, 1>;
        // x by way of LDS from five rows on: 2048 -> 4224 features at one row 6.2 us straight from x, 7.0 through LDS; 4864 -> 2048
        // features at eight rows 8.9 against 7.9
        if (n_rows <= 4 && x_is_f32 && share <= 16) by_share(bf_c, One{}, Yes{}, No{});
        else if (n_rows <= 4 && !x_is_f32) by_share(bf_c, One{}, No{}, No{});
        else if (x_is_f32 && nmb == 1) by_share(bf_c, One{}, Yes{}, Yes{});
        else if (x_is_f32) by_share(bf_c, integral_constant<int, 2>{}, Yes{}, Yes{});
        else if (nmb == 1) by_share(bf_c, One{}, No{}, Yes{});
        else if (nmb == 2) by_share(bf_c, integral_constant<int, 2>{}, No{}, Yes{});
        else if (nmb == 3) by_share(bf_c, integral_constant<int, 3>{}, No{}, Yes{});
        else by_share(bf_c, integral_constant<int, 4>{}, No{}, Yes{});
    };
    if (dtype == BITSMOE_DT_BF16) by_rows(Yes{}); else by_rows(No{});
    BITSMOE_HIP_TRY(hipGetLastError());
    return BITSMOE_OK;
}

// Prepared weights whose contraction is four whole shares of the few-rows kernel (hidden sizes 1024, 1536, 2048 and 2560), up to 128 experts.
bool bitsmoe::skinny_linear_takes_router(int64_t n_rows, int32_t in_features, int32_t weight_is_prepared, int32_t n_experts, int32_t top_k) {
    return n_rows >= 1 && n_rows <= 48 && weight_is_prepared != 0 && n_experts >= 1 && n_experts <= 128 && top_k >= 1 && top_k <= 64 && top_k <= n_experts &&
           (in_features == 1024 || in_features == 1536 || in_features == 2048 || in_features == 2560);
}

int bitsmoe::skinny_linear_with_router(const void* x, int32_t dtype, int64_t ld_x, const void* weight, int64_t n_rows, int32_t in_features,
                                       int32_t out_features, void* out, int64_t ld_out, const RouterBeside& router, void* stream) {
    BITSMOE_REQUIRE(dtype == BITSMOE_DT_F16 || dtype == BITSMOE_DT_BF16, "dtype must be f16 (0) or bf16 (1)");
    BITSMOE_REQUIRE(skinny_linear_takes_router(n_rows, in_features, 1, router.n_experts, router.top_k), "not a shape of the joint launch");
    BITSMOE_REQUIRE(out_features >= 2 && out_features % 2 == 0, "out_features must be even");
    BITSMOE_REQUIRE(ld_x >= in_features && ld_x % 8 == 0, "ld_x must be at least in_features and a multiple of 8");
    BITSMOE_REQUIRE(ld_out >= out_features && ld_out % 2 == 0, "ld_out must be at least out_features and even");
    BITSMOE_REQUIRE(router.round_dtype >= -1 && router.round_dtype <= 1, "round_dtype must be -1 (none), 0 (fp16) or 1 (bf16)");
    BITSMOE_REQUIRE(x && weight && out && router.weight && router.selected && router.weights, "null pointer");
    BITSMOE_REQUIRE((((uintptr_t)x | (uintptr_t)weight | (uintptr_t)router.weight) & 15) == 0 && ((uintptr_t)out & 3) == 0,
                    "x and the weights must be 16-byte aligned, out 4-byte aligned");
    const int router_blocks = (int)((n_rows + 3) / 4);
    const dim3 grid((unsigned)(router_blocks + (out_features + 15) / 16));
    auto run_nb = [&](auto bf_c, auto nmb_c, auto s_c, auto turn_c, auto nb_c) {
        hipLaunchKernelGGL((k_skinny_linear_router<decltype(bf_c)::value, decltype(nmb_c)::value, decltype(s_c)::value, decltype(turn_c)::value,
                                                   decltype(nb_c)::value>), grid, dim3(256), 0, (hipStream_t)stream, x, ld_x, (const uint16_t*)weight, (int)n_rows, in_features, out_features,
                           (uint16_t*)out, ld_out, router_blocks, router);
    };
    auto run = [&](auto bf_c, auto nmb_c, auto s_c, auto turn_c) {
        if (router.n_experts <= 64) run_nb(bf_c, nmb_c, s_c, turn_c, std::integral_constant<int, 4>{});
        else run_nb(bf_c, nmb_c, s_c, turn_c, std::integral_constant<int, 8>{});
    };
    auto by_share = [&](auto bf_c, auto nmb_c, auto turn_c) {
        if (in_features == 1024) run(bf_c, nmb_c, std::integral_constant<int, 8>{}, turn_c);
        else if (in_features == 1536) run(bf_c, nmb_c, std::integral_constant<int, 12>{}, turn_c);
        else if (in_features == 2048) run(bf_c, nmb_c, std::integral_constant<int, 16>{}, turn_c);
        else run(bf_c, nmb_c, std::integral_constant<int, 20>{}, turn_c);
    };
    auto by_rows = [&](auto bf_c) {
        if (n_rows <= 4) by_share(bf_c, std::integral_constant<int, 1>{}, std::false_type{});
        else if (n_rows <= 16) by_share(bf_c, std::integral_constant<int, 1>{}, std::true_type{});
        else if (n_rows <= 32) by_share(bf_c, std::integral_constant<int, 2>{}, std::true_type{});
        else by_share(bf_c, std::integral_constant<int, 3>{}, std::true_type{});
    };
    if (dtype == BITSMOE_DT_BF16) by_rows(std::true_type{}); else by_rows(std::false_type{});
    BITSMOE_HIP_TRY(hipGetLastError());
    return BITSMOE_OK;
}
