// A bias-free linear layer for MANY rows: out[M, N] = x[M, K] * W[N, K]^T, 16-bit x / W / out, fp32 sums.
// The two GEMMs around the routed-expert operator (skinny_linear.hip has their few-rows form; bitsmoe/models/qwen3moe/
// bitsmoe_block.py:63-64, bitsmoe/models/base_block.py:414) from decode batches of tens of tokens up to prompts of thousands.
// W is read in the framework's [out_features, in_features] layout.
//
// What bounds it: at most sizes neither the matrix cores nor HBM but what one CU can fetch, about 50 bytes a nanosecond when the
// weights come from memory (75 to 110 from the caches), however deep the ring.  So tiles are as square and as large as a
// launch that still fills 256 CUs allows, and the rule below looks for that.  The loads go straight into LDS and are issued one by one
// between the MFMAs: all of a stage at once they queue, and a wavefront that waits to issue a load issues no MFMA (a step of 64
// contraction indices of a 256 x 128 tile, one workgroup: 0.74 us with the loads at once, 0.56 spread; 64 x 64: 0.225 -> 0.147).
// us per launch, library GEMM of the framework -> this kernel with the tile the rule picks, graph over 300 MB of weights:
//   in -> out features    64 rows      128          256          512          1500         4096
//   2048 -> 4224       13.0 ->  9.6  15.0 -> 12.2  23.8 -> 14.8  23.3 -> 20.8  31.6 -> 29.3  80.6 -> 68.1
//   2048 -> 2048        8.9 ->  5.5   8.8 ->  5.7  10.1 ->  7.7  11.2 ->  9.2  18.6 -> 17.1  34.1 -> 31.8
//   2048 -> 9728       16.4 -> 14.6  18.2 -> 16.4  27.2 -> 21.1  30.2 -> 29.7  (library)    163 -> 148
//   4864 -> 2048       16.7 -> 13.8  14.9 -> 13.8  (library)     24.9 -> 24.1  (library)    73.8 -> 66.0
#include "common.h"
#include "lds_direct.h"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>

namespace bitsmoe {

typedef float tl_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t tl_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t tl_u32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 tl_f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 tl_bf16x8 __attribute__((ext_vector_type(8)));

// One workgroup = BM rows x BN columns, WM x WN wavefronts.  A stage holds KS slabs of 64 contraction indices of both operands;
// STAGES of them are in LDS or on their way there.  Rows past M or N repeat the last one and are not stored.
template <bool BF16, int BM, int BN, int WM, int WN, int KS, int STAGES, int PER_SIMD>
__global__ __launch_bounds__(64 * WM * WN, PER_SIMD) void k_tiled_linear(const uint16_t* __restrict__ x, int64_t ld_x,
                                                                         const uint16_t* __restrict__ w, int M, int K, int N,
                                                                         uint16_t* __restrict__ out, int64_t ld_out,
                                                                         const float* __restrict__ addend, int64_t ld_add,
                                                                         int m_tiles, int n_tiles) {
    constexpr int NW = WM * WN;
    constexpr int MB = BM / WM / 16, NB = BN / WN / 16;        // 16 x 16 blocks of a wavefront
    constexpr int XL = BM / 8 / NW, WL = BN / 8 / NW;          // load instructions per slab and wavefront
    static_assert(XL * NW * 8 == BM && WL * NW * 8 == BN && MB * WM * 16 == BM && NB * WN * 16 == BN && NW % 2 == 0, "whole pieces");
    constexpr int G = KS * (XL + WL);
    constexpr int SLAB = (BM + BN) * 64;                       // 16-bit elements
    __shared__ __attribute__((aligned(16))) uint16_t lds[STAGES * KS * SLAB];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wv / WN, wn = wv % WN;
    const int n = lane & 15, kg = lane >> 4;
    // Workgroup b runs on XCD b % 8, and every XCD has its own L2: each gets a consecutive eighth of the tiles, which walk over
    // the columns four row tiles at a time, so that the tiles an XCD works on at one time share their operands.
    const int total = m_tiles * n_tiles;
    const int per_xcd = (total + 7) / 8;
    const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || tile >= total) return;
    constexpr int GROUP = 4;
    const int group = tile / (GROUP * n_tiles), in_group = tile - group * (GROUP * n_tiles);
    const int group_rows = min(GROUP, m_tiles - group * GROUP);
    const int m0 = (group * GROUP + in_group % group_rows) * BM, n0 = (in_group / group_rows) * BN;

    // the chunk of its row that lands at this lane's place (every load of a wavefront starts at a multiple of 8 rows)
    const int l3 = lane >> 3;
    const uint32_t chunk = (uint32_t)(((lane & 7) ^ (4 * (wv & 1) + (l3 >> 1))) * 16);
    const unsigned char* xb = (const unsigned char*)(x + (int64_t)m0 * ld_x);
    const unsigned char* wb = (const unsigned char*)(w + (int64_t)n0 * K);
    uint32_t xo[XL], wo[WL];
#pragma unroll
    for (int i = 0; i < XL; ++i) xo[i] = (uint32_t)min((i * NW + wv) * 8 + l3, M - 1 - m0) * (uint32_t)(ld_x * 2) + chunk;
#pragma unroll
    for (int i = 0; i < WL; ++i) wo[i] = (uint32_t)min((i * NW + wv) * 8 + l3, N - 1 - n0) * (uint32_t)(K * 2) + chunk;
    const uint32_t lds_at = lds_address(lds);
    auto request_piece = [&](auto l_c, int step, int stage) {
        constexpr int L = decltype(l_c)::value, Q = L / (XL + WL), I = L % (XL + WL);
        const uint32_t at = lds_at + 2 * (stage * (KS * SLAB) + wv * 512 + Q * SLAB);
        const int64_t k = ((int64_t)step * KS + Q) * 128;
        if constexpr (I < XL)
            load_to_lds16(xb + k, xo[I], at + 2 * (I * NW * 512));
        else
            load_to_lds16(wb + k, wo[I - XL], at + 2 * (BM * 64 + (I - XL) * NW * 512));
    };
    tl_f32x4 acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = tl_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](tl_f32x4& c, tl_u32x4 bv, tl_u32x4 av) {
        if constexpr (BF16)
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(tl_bf16x8, bv), __builtin_bit_cast(tl_bf16x8, av), c, 0, 0, 0);
        else
            c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(tl_f16x8, bv), __builtin_bit_cast(tl_f16x8, av), c, 0, 0, 0);
    };
    const int steps = K / (64 * KS);
    // at most `later` stages may still be on their way
    auto landed = [&](int later) {
        if (later <= 0) wait_vmcnt<0>();
        static_for([&](auto l_c) {
            if (later == decltype(l_c)::value + 1) wait_vmcnt<(decltype(l_c)::value + 1) * G>();
        }, std::make_integer_sequence<int, STAGES - 1>{});
    };
    for (int s = 0; s < min(steps, STAGES); ++s) static_for([&](auto l_c) { request_piece(l_c, s, s); }, std::make_integer_sequence<int, G>{});
    landed(min(steps, STAGES) - 1);
    barrier_no_drain();
    const int lane_a = (wm * MB * 16 + n) * 64, lane_b = BM * 64 + (wn * NB * 16 + n) * 64;
    tl_u32x4 a[MB], b[2][NB];
    // A phase is 32 contraction indices.  The operands of a phase are read while the MFMAs of the one before run, a row block's as
    // soon as its last MFMA has been issued.
    constexpr int PHASES = 2 * KS;
    auto at_phase = [&](int stage, int u) { return lds + stage * (KS * SLAB) + (u / 2) * SLAB + (((4 * (u & 1) + kg) ^ (n >> 1)) << 3); };
    // phase U of the stage at hand; reads phase (U + 1) % PHASES from `from`.  REQUEST: the loads of step `step` are issued between the
    // MFMAs of the PHASES phases from a stage's last one on.  (All at once they keep a wavefront from its MFMAs while they queue.)
    auto phase = [&](auto u_c, auto request_c, const uint16_t* from, int step, int stage) {
        constexpr int U = decltype(u_c)::value;
        constexpr int TURN = (U + 1) % PHASES;      // 0: the last phase
#pragma unroll
        for (int j = 0; j < NB; ++j) b[(U + 1) & 1][j] = *reinterpret_cast<const tl_u32x4*>(from + lane_b + j * 1024);
        static_for([&](auto i_c) {
            constexpr int I = decltype(i_c)::value;
            if constexpr (decltype(request_c)::value) {
                constexpr int SLOT = TURN * MB + I, FIRST = (SLOT * G + PHASES * MB - 1) / (PHASES * MB),
                              END = ((SLOT + 1) * G + PHASES * MB - 1) / (PHASES * MB);
                static_for([&](auto l_c) { request_piece(std::integral_constant<int, FIRST + decltype(l_c)::value>{}, step, stage); },
                           std::make_integer_sequence<int, END - FIRST>{});
            }
#pragma unroll
            for (int j = 0; j < NB; ++j) multiply(acc[I][j], b[U & 1][j], a[I]);
            a[I] = *reinterpret_cast<const tl_u32x4*>(from + lane_a + I * 1024);
            // (left alone, the compiler gathers the MFMAs in front of the barrier, and every operand is waited for where it is used)
            __builtin_amdgcn_sched_barrier(0);
        }, std::make_integer_sequence<int, MB>{});
    };
#pragma unroll
    for (int j = 0; j < NB; ++j) b[0][j] = *reinterpret_cast<const tl_u32x4*>(at_phase(0, 0) + lane_b + j * 1024);
#pragma unroll
    for (int i = 0; i < MB; ++i) a[i] = *reinterpret_cast<const tl_u32x4*>(at_phase(0, 0) + lane_a + i * 1024);
    int stage = 0;
    auto inner_phases = [&](auto request_c, int now, int step, int into) {
        static_for([&](auto u_c) { phase(u_c, request_c, at_phase(now, decltype(u_c)::value + 1), step, into); },
                   std::make_integer_sequence<int, PHASES - 1>{});
    };
    using Last = std::integral_constant<int, PHASES - 1>;
    inner_phases(std::false_type{}, 0, 0, 0);
    // From the last phase of step s to the one before the last of step s + 1.  When the last phase of a stage begins, every wavefront
    // has read all of the stage: there the next stage is waited for, and a new one goes into this one's place.
    auto round = [&](auto request_c, int s, int later) {
        wait_lds_reads();
        landed(later);
        barrier_no_drain();
        const int next = stage == STAGES - 1 ? 0 : stage + 1;
        phase(Last{}, request_c, at_phase(next, 0), s + STAGES, stage);
        inner_phases(request_c, next, s + STAGES, stage);
        stage = next;
    };
    int s = 0;
    for (; s < steps - STAGES; ++s) round(std::true_type{}, s, STAGES - 2);
    for (; s < steps - 1; ++s) round(std::false_type{}, s, min(steps - 2 - s, STAGES - 2));
    phase(Last{}, std::false_type{}, at_phase(stage, 0), 0, 0);      // (what it reads is not used)
    // W is the MFMA's first operand: a lane holds columns 16 j + 4 kg .. + 3 of row 16 i + n
    auto round16 = [](float v) -> uint32_t {
        if constexpr (BF16)
            return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)v);
        else
            return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v);
    };
    const int row0 = m0 + wm * MB * 16, col0 = n0 + wn * NB * 16;
    auto rounded = [&](tl_f32x4 v) { return tl_u32x2{round16(v[0]) | (round16(v[1]) << 16), round16(v[2]) | (round16(v[3]) << 16)}; };
    auto add_row = [&](int i) {      // (fp32 [M, N] added to the sums before the one rounding of the result)
        const float* from = addend + (int64_t)min(row0 + 16 * i + n, M - 1) * ld_add;
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] += *reinterpret_cast<const tl_f32x4*>(from + min(col0 + 16 * j + 4 * kg, N - 4));
    };
    if constexpr (NB == 4) {
        // turned around in LDS, so that a store instruction writes eight whole rows of 128 bytes
        wait_lds_reads();
        barrier_no_drain();
        uint16_t* turn = lds + wv * (MB * 16 * 64);
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            if (addend) add_row(i);
#pragma unroll
            for (int j = 0; j < NB; ++j)
                *reinterpret_cast<tl_u32x2*>(turn + dma_chunk_off(16 * i + n, 2 * j + (kg >> 1)) + 4 * (kg & 1)) = rounded(acc[i][j]);
        }
#pragma unroll
        for (int k = 0; k < 2 * MB; ++k) {
            const int r = 8 * k + l3, col = col0 + 8 * (lane & 7);
            if (row0 + r < M && col < N)
                *reinterpret_cast<tl_u32x4*>(out + (int64_t)(row0 + r) * ld_out + col) =
                    *reinterpret_cast<const tl_u32x4*>(turn + dma_chunk_off(r, lane & 7));
        }
    } else {
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            if (addend) add_row(i);
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                const int row = row0 + 16 * i + n, col = col0 + 16 * j + 4 * kg;
                if (row < M && col < N) *reinterpret_cast<tl_u32x2*>(out + (int64_t)row * ld_out + col) = rounded(acc[i][j]);
            }
        }
    }
}

}  // namespace bitsmoe

using namespace bitsmoe;

// ---- which tile, and whether at all ------------------------------------------------------------------------------------
// us per 64 contraction indices: `one` for a launch of at most 256 tiles (one per CU), `more` for every further 256.  Tiles of which
// a CU holds several overlap, so there the second round is counted by its share; the others in whole rounds.  Measured at 2048 -> 4224,
// 5640 and 9728 features, 64 to 4096 rows, weights from memory.
namespace {
struct Tile {
    int rows, cols;
    double one, more;
    bool shared;      // several workgroups per CU
    bool single;      // only in launches of at most one round (128 x 192 in two rounds: 2048 -> 5640 at 2048 rows 53.2 us, library 50.3)
    // Where the tile is the faster one, next to the framework's GEMM (tiled_linear_pays below): contractions of up to `k_filled` in one round
    // that takes at least `filled` of the CUs, of up to `k_emptier` in an emptier one, of up to `k_more` in more than one round (`shared` only).
    double filled;
    int k_filled, k_emptier, k_more;
};
constexpr int ANY_K = 1 << 22;
constexpr Tile TILES[] = {
    {256, 160, 1.15, 1.15, false, false, 0.75, ANY_K, 0, 0},   {256, 128, 0.90, 0.90, false, false, 0.75, ANY_K, 0, 0},
    {192, 192, 1.06, 1.06, false, false, 0.70, ANY_K, 0, 0},   {128, 192, 0.84, 0.84, false, true, 0.80, ANY_K, 2048, 0},
    {128, 128, 0.62, 0.62, false, false, 0.80, ANY_K, 2048, 0}, {128, 96, 0.60, 0.60, false, false, 0.70, ANY_K, 0, 0},
    {128, 64, 0.52, 0.55, true, false, 0.80, ANY_K, 1536, 1024}, {64, 96, 0.46, 0.46, false, false, 0.60, ANY_K, 0, 0},
    {64, 64, 0.41, 0.40, true, false, 0.0, 6144, 0, 1536},     {64, 32, 0.36, 0.30, true, false, 0.0, 4096, 0, 4096},
    {32, 32, 0.31, 0.20, true, false, 0.60, ANY_K, 5120, 5120},
};
constexpr int N_TILES_KNOWN = sizeof(TILES) / sizeof(TILES[0]);
constexpr int CUS = 256;

int64_t tiles_of(const Tile& t, int64_t rows, int out_features) {
    return ((rows + t.rows - 1) / t.rows) * ((out_features + t.cols - 1) / t.cols);
}

int best_tile(int64_t rows, int out_features) {
    int best = -1;
    double least = 0.0;
    for (int i = 0; i < N_TILES_KNOWN; ++i) {
        const Tile& t = TILES[i];
        const double rounds = (double)tiles_of(t, rows, out_features) / CUS;
        if (t.single && rounds > 1.0) continue;
        const double cost = t.one + t.more * (t.shared ? std::max(0.0, rounds - 1.0) : std::max(0.0, std::ceil(rounds) - 1.0));
        if (best < 0 || cost < least) best = i, least = cost;
    }
    return best;
}
}  // namespace

// Is this kernel the faster one, next to the framework's GEMM?  That one may split the contraction, cuts its tiles to fit and has
// tiles of 256 x 256; this one does neither, so it depends on the tile, on the share of the CUs' places that a launch takes and, in
// emptier launches, on the contraction.  Time over the framework's, medians over cold weights, 5980 shapes of 49 to 8192
// rows, 128 to 8192 and 64 to 12288 features (means of a band; of the 4946 shapes that get a yes 65 are above 1.03, the worst 1.23; of
// the others the worst 1.68):
//   32 x 32, less than 0.6 of the CUs:  up to 5120 in features 0.3 to 0.9, from 6144 on 1.03 to 1.16;  fuller: 0.5 to 0.96 at all
//   64 x 32:  up to 4096 0.6 to 0.93, 5120 0.94 to 1.02, longer 0.9 to 1.09
//   64 x 64:  one round 0.6 to 0.98 up to 6144; two: 1024 0.75, 1536 0.78, 2048 0.94 (up to 272 tiles 0.89, 288 1.01), 2560 0.99, 4096 1.01
//   128 x 64: one round of 0.8 or more 0.6 to 1.0 at all, emptier 0.7 to 0.8 up to 1536 and 1.06 to 1.13 longer; two: 1024 0.88, 2048 0.97
//             (0.83 to 1.37), longer 1.07 to 1.17
//   128 x 128, 128 x 192: 0.8 or more 0.65 to 0.99, emptier 0.74 to 0.97 up to 2048 and 0.95 to 1.07 longer
//   the others in one round 0.6 to 0.98
// Several rounds of a tile that a CU holds one of: 0.5 to 1.02 where at least 0.93 of the last one is taken, 0.96 to 1.27 when 0.86 or 0.89
// are; but 1.04 to 1.2 where tiles of 256 x 256 fill the CUs about as well (4096 x 7168, 3546 x 4608, 3909 x 4096).
extern "C" int32_t bitsmoe_tiled_linear_pays(int64_t n_rows, int32_t in_features, int32_t out_features) {
    if (n_rows <= 0 || in_features < 128 || in_features > (1 << 22) || in_features % 128 != 0 || out_features < 8 || out_features % 8 != 0) return 0;
    const Tile& t = TILES[best_tile(n_rows, out_features)];
    auto taken = [](int64_t tiles) { return (double)tiles / (double)((tiles + CUS - 1) / CUS * CUS); };
    const int64_t tiles = tiles_of(t, n_rows, out_features);
    if (tiles <= CUS) return in_features <= (taken(tiles) >= t.filled ? t.k_filled : t.k_emptier);
    // (64 x 64 with at most a sixteenth more than one round: up to 2048)
    if (t.shared) return in_features <= (t.rows == 64 && t.cols == 64 && tiles <= CUS + CUS / 16 ? 2048 : t.k_more);
    const int64_t of_256 = ((n_rows + 255) / 256) * ((out_features + 255) / 256);
    return taken(tiles) >= 0.93 && taken(of_256) < 0.85;
}

// The tile that the rule takes: its rows and columns (0: no size of the kernel's).
extern "C" int32_t bitsmoe_tiled_linear_tile(int64_t n_rows, int32_t out_features, int32_t* tile_rows, int32_t* tile_cols) {
    if (n_rows <= 0 || out_features < 8 || out_features % 8 != 0 || !tile_rows || !tile_cols) return 0;
    const Tile& t = TILES[best_tile(n_rows, out_features)];
    *tile_rows = t.rows;
    *tile_cols = t.cols;
    return 1;
}

extern "C" int bitsmoe_tiled_linear(const void* x, int32_t dtype, int64_t ld_x, const void* weight, int64_t n_rows, int32_t in_features,
                                    int32_t out_features, void* out, int64_t ld_out, const float* addend, int64_t ld_addend, void* stream) {
    BITSMOE_REQUIRE(dtype == BITSMOE_DT_F16 || dtype == BITSMOE_DT_BF16, "dtype must be f16 (0) or bf16 (1)");
    BITSMOE_REQUIRE(n_rows >= 0 && n_rows < ((int64_t)1 << 31) - 256, "n_rows must be in [0, 2^31 - 256)");
    BITSMOE_REQUIRE(in_features >= 128 && in_features % 128 == 0, "in_features must be a positive multiple of 128");
    BITSMOE_REQUIRE(out_features >= 8 && out_features % 8 == 0, "out_features must be a positive multiple of 8");
    // (a tile's rows are addressed by 32 bits of byte offset from its first one)
    BITSMOE_REQUIRE(ld_x >= in_features && ld_x % 8 == 0 && ld_x <= (1 << 22) && in_features <= (1 << 22),
                    "ld_x must be at least in_features, a multiple of 8 and at most 2^22");
    BITSMOE_REQUIRE(ld_out >= out_features && ld_out % 8 == 0, "ld_out must be at least out_features and a multiple of 8");
    BITSMOE_REQUIRE(addend == nullptr || (ld_addend >= out_features && ld_addend % 4 == 0), "ld_addend must be at least out_features and a multiple of 4");
    if (n_rows == 0) return BITSMOE_OK;
    BITSMOE_REQUIRE(x && weight && out, "null pointer");
    BITSMOE_REQUIRE((((uintptr_t)x | (uintptr_t)weight | (uintptr_t)out | (uintptr_t)addend) & 15) == 0,
                    "x, weight, out and addend must be 16-byte aligned");
    const int chosen = best_tile(n_rows, out_features);
    BITSMOE_REQUIRE(tiles_of(TILES[chosen], n_rows, out_features) < ((int64_t)1 << 30), "too many rows");
    hipStream_t st = (hipStream_t)stream;
    // wavefronts over rows and columns, slabs per stage, stages, wavefronts per SIMD
    auto launch = [&](auto bf_c, auto i_c, auto wm_c, auto wn_c, auto ks_c, auto stages_c, auto per_simd_c) {
        constexpr Tile t = TILES[decltype(i_c)::value];
        constexpr int WM = decltype(wm_c)::value, WN = decltype(wn_c)::value;
        const int mt = (int)((n_rows + t.rows - 1) / t.rows), nt = (out_features + t.cols - 1) / t.cols;
        hipLaunchKernelGGL((k_tiled_linear<decltype(bf_c)::value, t.rows, t.cols, WM, WN, decltype(ks_c)::value, decltype(stages_c)::value,
                                           decltype(per_simd_c)::value>),
                           dim3((unsigned)((mt * nt + 7) / 8 * 8)), dim3(64 * WM * WN), 0, st, (const uint16_t*)x, ld_x, (const uint16_t*)weight,
                           (int)n_rows, in_features, out_features, (uint16_t*)out, ld_out, addend, ld_addend, mt, nt);
    };
    auto run = [&](auto bf_c) {
        using std::integral_constant;
        const integral_constant<int, 1> one;
        const integral_constant<int, 2> two;
        const integral_constant<int, 3> three;
        const integral_constant<int, 4> four;
        const integral_constant<int, 5> five;
        switch (chosen) {
            case 0: return launch(bf_c, integral_constant<int, 0>{}, two, two, one, three, one);
            case 1: return launch(bf_c, integral_constant<int, 1>{}, two, two, one, three, one);
            case 2: return launch(bf_c, integral_constant<int, 2>{}, two, four, one, three, two);
            case 3: return launch(bf_c, integral_constant<int, 3>{}, two, two, one, three, one);
            case 4: return launch(bf_c, integral_constant<int, 4>{}, two, two, one, four, one);
            case 5: return launch(bf_c, integral_constant<int, 5>{}, two, two, one, five, one);
            case 6: return launch(bf_c, integral_constant<int, 6>{}, two, two, one, three, two);
            case 7: return launch(bf_c, integral_constant<int, 7>{}, two, two, one, five, one);
            case 8: return launch(bf_c, integral_constant<int, 8>{}, two, two, one, four, two);
            case 9: return launch(bf_c, integral_constant<int, 9>{}, four, one, one, four, three);
            default: return launch(bf_c, integral_constant<int, 10>{}, two, two, two, four, two);
        }
    };
    if (dtype == BITSMOE_DT_BF16) run(std::true_type{}); else run(std::false_type{});
    BITSMOE_HIP_TRY(hipGetLastError());
    return BITSMOE_OK;
}
