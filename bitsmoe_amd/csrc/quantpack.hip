// The quantiser that defines the payload's contents and the slab packer, as kernels.
//
//   k_quantize_tiles   sixteen lanes per (row, 128-column tile): the symmetric quantiser of
//                      bitsmoe/quant/quantizer.py:30-84 -- 2/3/4 bits: scale_0 = mean|x|, then `iters` times
//                      { q = clamp(round_half_even(x / scale)); scale = max(mean(x q) / (mean(q q) + eps), eps) }
//                      with the means over the tile's real columns; 6/8 bits: absmax; 1 bit: sign, mean|x|.
//                      The levels returned are those of the last pass, the scale the one fitted to them.
//   k_pack_slabs       levels of one bit bucket -> payload words in the runtime order
//                      [slab of <= 64 rows][tile][stage of 16 rows][micro of 32 columns][row][plane]
//                      (bitsmoe/quant/packer.py:169-306) and scales in [slab][tile][row] order; the plane
//                      words come from wave64 ballots, two 32-column micro-tiles per wavefront.
//   k_pack_matrix      both of them for a whole matrix with rows of several widths (rows gathered by ranges, 16-bit rows
//                      stored as they are), and its tables, in one launch.
//
// Sums run over the lanes in a fixed order that differs from the framework's reduction order, so a
// scale can differ from the CPU restatement's in its last bit and a level with it where x / scale sits
// on a rounding tie; given equal levels the words are identical.
#include <algorithm>

#include "common.h"

namespace bitsmoe {

// ---- the quantiser of one tile over sixteen lanes ----------------------------------------------------------------------
// Lane j of the group holds columns j + 16 m, m = 0..7.  The iteration is bound by vector instructions (its data stays in
// registers), so the layout is the one with the fewest of them: four tiles per wavefront share every instruction, the last
// four of the seven summation steps are row rotations that ride in the adds (with one tile per wavefront all but one step
// went through the LDS crossbar: six dependent permutes per sum), and the quotient x / scale is the product with one
// reciprocal per tile and pass wherever that settles the rounding.  The iteration ends early once a pass leaves every scale
// of the wavefront as it was: the remaining passes would repeat it.  Same values, bit for bit, as one tile per wavefront with
// all divisions and passes.  1978 x 1408 values in three widths: 173 us in three launches that way and 16 us for the
// packer's three, 24 us for both in the one launch of k_pack_matrix.
template <int N>
__device__ __forceinline__ float row_ror(float v) {      // the value of the lane N places away inside the row of sixteen
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), 0x120 + N, 0xF, 0xF, false));
}
__device__ __forceinline__ float row_sum16(float v) {
    v += row_ror<8>(v);
    v += row_ror<4>(v);
    v += row_ror<2>(v);
    return v + row_ror<1>(v);
}
__device__ __forceinline__ float row_max16(float v) {
    v = fmaxf(v, row_ror<8>(v));
    v = fmaxf(v, row_ror<4>(v));
    v = fmaxf(v, row_ror<2>(v));
    return fmaxf(v, row_ror<1>(v));
}
// Sum over a tile of terms that are already added in pairs (columns c and c + 64): p[m] is the pair of column j + 16 m.
__device__ __forceinline__ float tile_sum(const float (&p)[4]) { return row_sum16((p[0] + p[2]) + (p[1] + p[3])); }

struct TileLevels {
    float q[8];
    float scale;
};

// levels of x / scale for a lane's eight columns, as clamp(rint(x / scale)) with the correctly rounded quotient gives them.
// t = x * (1 / scale) is within 2^-23 of the quotient (relative); where t is not that close to a half-integer both round
// alike (beyond the clamp's ends it does not matter), else the lane divides.
__device__ __forceinline__ void round_levels(const float (&x)[8], float scale, float lo, float hi, float (&q)[8]) {
    const float inv = 1.0f / scale;
    bool unsure = !(scale < 1e37f);      // (the reciprocal would lose bits)
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        const float t = x[m] * inv;
        q[m] = rintf(t);
        unsure |= fabsf(t - q[m]) > 0.49999f;
    }
    if (unsure) {
#pragma unroll
        for (int m = 0; m < 8; ++m) q[m] = rintf(x[m] / scale);
    }
#pragma unroll
    for (int m = 0; m < 8; ++m) q[m] = fminf(fmaxf(q[m], lo), hi);
}

// x: a lane's columns (0 past n_valid); j = lane % 16.
__device__ __forceinline__ TileLevels quantize_tile(const float (&x)[8], int j, int n_valid, int bits, int iters, float eps) {
    TileLevels r;
    const float lo = -(float)(1 << (bits - 1)), hi = (float)((1 << (bits - 1)) - 1);
    const float inv_n = 1.0f / (float)n_valid;
    const bool tail = n_valid < N_TILE;
    auto drop_tail = [&]() {      // (a column past the end counts for nothing, whatever the scale is)
        if (tail)
#pragma unroll
            for (int m = 0; m < 8; ++m)
                if (j + 16 * m >= n_valid) r.q[m] = 0.0f;
    };
    if (bits > 4) {
        float mx = 0.0f;
#pragma unroll
        for (int m = 0; m < 8; ++m) mx = fmaxf(mx, fabsf(x[m]));
        r.scale = fmaxf(row_max16(mx) / hi, eps);
        round_levels(x, r.scale, lo, hi, r.q);
        drop_tail();
        return r;
    }
    float p[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) p[m] = fabsf(x[m]) + fabsf(x[m + 4]);
    r.scale = fmaxf(tile_sum(p) * inv_n, eps);
    if (bits == 1) {
#pragma unroll
        for (int m = 0; m < 8; ++m) r.q[m] = x[m] < 0.0f ? -1.0f : 1.0f;
        drop_tail();
        return r;
    }
    for (int it = 0; it < iters; ++it) {
        round_levels(x, r.scale, lo, hi, r.q);
        drop_tail();
        float g[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            p[m] = __builtin_fmaf(x[m], r.q[m], x[m + 4] * r.q[m + 4]);
            g[m] = __builtin_fmaf(r.q[m], r.q[m], r.q[m + 4] * r.q[m + 4]);
        }
        const float xq = tile_sum(p) * inv_n;
        const float qq = __builtin_fmaf(inv_n, tile_sum(g), eps);
        const float next = fmaxf(xq / qq, eps);
        const bool moved = __float_as_uint(next) != __float_as_uint(r.scale);
        r.scale = next;
        if (__ballot(moved) == 0) break;
    }
    return r;
}

// A lane's columns of tile t of a row (0 past the row's end).
__device__ __forceinline__ void load_tile16(const float* __restrict__ row, int64_t dim, int t, int j, float (&x)[8]) {
    const int n_valid = (int)min((int64_t)N_TILE, dim - (int64_t)t * N_TILE);
    const float* src = row + (int64_t)t * N_TILE;
#pragma unroll
    for (int m = 0; m < 8; ++m) x[m] = j + 16 * m < n_valid ? src[j + 16 * m] : 0.0f;
}

// grid-stride over (row, tile) units, sixteen lanes each.
__global__ __launch_bounds__(256) void k_quantize_tiles(const float* __restrict__ rows, int64_t k, int64_t dim,
                                                        int64_t row_stride, int n_tiles, int bits, int iters, float eps,
                                                        int8_t* __restrict__ levels, float* __restrict__ scale_out) {
    const int j = threadIdx.x & 15;
    const int64_t n_units = k * n_tiles;
    const int64_t first = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 4;
    const int64_t step = ((int64_t)gridDim.x * blockDim.x) >> 4;
    for (int64_t unit = first; unit < n_units; unit += step) {
        const int64_t row = unit / n_tiles;
        const int t = (int)(unit - row * n_tiles);
        float x[8];
        load_tile16(rows + row * row_stride, dim, t, j, x);
        const TileLevels r = quantize_tile(x, j, (int)min((int64_t)N_TILE, dim - (int64_t)t * N_TILE), bits, iters, eps);
        // levels are stored over whole tiles: padding columns hold level 0
        int8_t* dst = levels + (row * n_tiles + t) * N_TILE;
#pragma unroll
        for (int m = 0; m < 8; ++m) dst[j + 16 * m] = (int8_t)r.q[m];
        if (j == 0) scale_out[row * n_tiles + t] = r.scale;
    }
}

__device__ inline unsigned code_of_level(int q, int bits) {
    return (bits == 1) ? (unsigned)((q + 1) >> 1) : (unsigned)(q + level_offset(bits));
}

// levels int8 [k, n_tiles * 128] of ONE bit bucket (rows in bucket order), scale fp32 [k, n_tiles] ->
// payload words and fp16 scales of the bucket's slabs (slab i = rows [64 i, 64 i + 64), the last one ragged).
// One wavefront per (row, tile, micro pair).
__global__ __launch_bounds__(256) void k_pack_slabs(const int8_t* __restrict__ levels, const float* __restrict__ scale,
                                                    int64_t k, int n_tiles, int bits, uint32_t* __restrict__ payload,
                                                    __half* __restrict__ scale_out) {
    const int lane = threadIdx.x & 63;
    const int64_t n_units = k * n_tiles * 2;
    const int64_t wave0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t n_waves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    const int w = bits;
    for (int64_t unit = wave0; unit < n_units; unit += n_waves) {
        const int half = (int)(unit & 1);
        const int64_t rt = unit >> 1;
        const int64_t row = rt / n_tiles;
        const int t = (int)(rt - row * n_tiles);
        const int64_t slab = row / K_SLAB;
        const int r_in = (int)(row - slab * K_SLAB);
        const int k_slab = (int)min((int64_t)K_SLAB, k - slab * K_SLAB);
        const int stage = r_in / K_STAGE, rr = r_in - stage * K_STAGE;
        const int rows_cur = min(K_STAGE, k_slab - stage * K_STAGE);
        // words before this slab: full slabs of 64 rows; inside: tile, stage, micro, row, plane
        const int64_t slab_base = slab * (int64_t)K_SLAB * n_tiles * MICROS * w;
        const int64_t tile_base = slab_base + (int64_t)t * k_slab * MICROS * w + (int64_t)stage * K_STAGE * MICROS * w;
        const unsigned code = code_of_level((int)levels[(row * n_tiles + t) * N_TILE + half * 64 + lane], bits) & 0xFFu;
        for (int p = 0; p < w; ++p) {
            const uint64_t bal = __ballot((code >> p) & 1u);
            if (lane == 0) {
                const int m0 = half * 2;
                payload[tile_base + (int64_t)m0 * rows_cur * w + rr * w + p] = (uint32_t)(bal & 0xFFFFFFFFull);
                payload[tile_base + (int64_t)(m0 + 1) * rows_cur * w + rr * w + p] = (uint32_t)(bal >> 32);
            }
        }
        if (half == 0 && lane == 0)
            scale_out[slab * (int64_t)K_SLAB * n_tiles + (int64_t)t * k_slab + r_in] = __float2half(scale[row * n_tiles + t]);
    }
}

// ---- a whole matrix: rows of several widths, quantised, packed and described in one launch ------------------------------
constexpr int PACK_MAX_RANGES = 64;
constexpr int PACK_MAX_BUCKETS = 8;
// Rows [src, src + rows of the range) of the source are packed rows first ...; ranges of one width follow each other.
struct PackRange {
    int32_t first, src, bucket;
};
// The rows of one width: packed rows row0 ..., their words, scales and slabs from these offsets on.
struct PackBucket {
    int64_t pay_off, scale_off;
    int32_t bits, row0, rows, slab0;
};
struct PackTables {
    PackRange range[PACK_MAX_RANGES];
    PackBucket bucket[PACK_MAX_BUCKETS];
    int32_t n_ranges, n_buckets, row_end, n_slabs;      // this launch packs rows [range[0].first, row_end)
};

template <int SB>      // bytes of an element of s: 2 (f16), 4 (f32)
__global__ __launch_bounds__(256) void k_pack_matrix(const float* __restrict__ src, int64_t row_stride, int64_t dim, int n_tiles,
                                                     const void* __restrict__ s, const PackTables tab, int iters, float eps,
                                                     int unit_blocks, uint32_t* __restrict__ payload, __half* __restrict__ scale_out,
                                                     __half* __restrict__ s_out, int32_t* __restrict__ rank_idx,
                                                     int32_t* __restrict__ tile_meta, int32_t* __restrict__ slab_meta) {
    const int row_begin = tab.range[0].first;
    auto range_of = [&](int row) {
        int i = 0;
        for (int k = 1; k < tab.n_ranges; ++k) i = row >= tab.range[k].first ? k : i;
        return i;
    };
    if ((int)blockIdx.x >= unit_blocks) {
        // tables: one thread per packed row of this launch, then (the launch that brings slab_meta) per slab and tile
        int64_t i = (int64_t)((int)blockIdx.x - unit_blocks) * 256 + threadIdx.x;
        const int n_rows = tab.row_end - row_begin;
        if (i < n_rows) {
            const int row = row_begin + (int)i;
            const PackRange r = tab.range[range_of(row)];
            const int from = r.src + row - r.first;
            rank_idx[row] = from;
            s_out[row] = SB == 2 ? ((const __half*)s)[from] : __float2half(((const float*)s)[from]);
            return;
        }
        i -= n_rows;
        if (slab_meta == nullptr || i >= (int64_t)tab.n_slabs * n_tiles) return;
        const int slab = (int)(i / n_tiles), t = (int)(i - (int64_t)slab * n_tiles);
        int b = 0;
        for (int k = 1; k < tab.n_buckets; ++k) b = slab >= tab.bucket[k].slab0 ? k : b;
        const PackBucket bk = tab.bucket[b];
        const int in_bucket = slab - bk.slab0;
        const int k_slab = min(K_SLAB, bk.rows - in_bucket * K_SLAB);
        const int w = words_per_row(bk.bits);
        int32_t* tm = tile_meta + i * 3;
        tm[0] = (int32_t)(bk.pay_off + (int64_t)in_bucket * K_SLAB * MICROS * w * n_tiles + (int64_t)t * k_slab * MICROS * w);
        tm[1] = (int32_t)(bk.scale_off + (int64_t)in_bucket * K_SLAB * n_tiles + (int64_t)t * k_slab);
        tm[2] = (int32_t)min((int64_t)N_TILE, dim - (int64_t)t * N_TILE);
        if (t == 0) {
            int32_t* sm = slab_meta + (int64_t)slab * 4;
            sm[0] = bk.bits;
            sm[1] = k_slab;
            sm[2] = bk.row0 + in_bucket * K_SLAB;
            sm[3] = slab * n_tiles;
        }
        return;
    }
    const int j = threadIdx.x & 15, group = (threadIdx.x >> 4) & 3;      // group of sixteen lanes inside the wavefront
    const int64_t n_units = (int64_t)(tab.row_end - row_begin) * n_tiles;
    for (int64_t unit = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 4; unit < n_units; unit += (int64_t)unit_blocks * 16) {
        const int row = row_begin + (int)(unit / n_tiles);
        const int t = (int)(unit % n_tiles);
        const PackRange r = tab.range[range_of(row)];
        const PackBucket bk = tab.bucket[r.bucket];
        float x[8];
        load_tile16(src + (int64_t)(r.src + row - r.first) * row_stride, dim, t, j, x);
        const int in_bucket = row - bk.row0;
        const int slab = in_bucket / K_SLAB, r_in = in_bucket % K_SLAB;
        const int k_slab = min(K_SLAB, bk.rows - slab * K_SLAB);
        const int stage = r_in / K_STAGE, rr = r_in % K_STAGE;
        const int rows_cur = min(K_STAGE, k_slab - stage * K_STAGE);
        const int w = words_per_row(bk.bits);
        uint32_t* words = payload + bk.pay_off + (int64_t)slab * K_SLAB * n_tiles * MICROS * w + (int64_t)t * k_slab * MICROS * w +
                          (int64_t)stage * K_STAGE * MICROS * w;
        auto place = [&](int micro, int plane) { return micro * rows_cur * w + rr * w + plane; };
        float tile_scale = 1.0f;
        if (bk.bits == 16) {
            // halves as they are, two columns to a word: columns 2c and 2c + 1 of a micro-tile come from neighbouring lanes
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const uint32_t mine = __half_as_ushort(__float2half(x[m]));
                const uint32_t next = (uint32_t)__shfl_down((int)mine, 1);
                if ((j & 1) == 0) words[place(m >> 1, 8 * (m & 1) + (j >> 1))] = mine | (next << 16);
            }
        } else {
            const TileLevels q = quantize_tile(x, j, (int)min((int64_t)N_TILE, dim - (int64_t)t * N_TILE), bk.bits, iters, eps);
            tile_scale = q.scale;
            unsigned code[8];
#pragma unroll
            for (int m = 0; m < 8; ++m) code[m] = code_of_level((int)q.q[m], bk.bits) & 0xFFu;
            // plane words: sixteen bits of a ballot are one half of a micro-tile's 32 columns
            for (int p = 0; p < w; ++p) {
#pragma unroll
                for (int micro = 0; micro < MICROS; ++micro) {
                    const uint64_t lo = __ballot((code[2 * micro] >> p) & 1u), hi = __ballot((code[2 * micro + 1] >> p) & 1u);
                    const uint32_t word = (uint32_t)((lo >> (16 * group)) & 0xFFFFu) | ((uint32_t)((hi >> (16 * group)) & 0xFFFFu) << 16);
                    if (j == micro) words[place(micro, p)] = word;
                }
            }
        }
        if (j == 0) scale_out[bk.scale_off + (int64_t)slab * K_SLAB * n_tiles + (int64_t)t * k_slab + r_in] = __float2half(tile_scale);
    }
}

}  // namespace bitsmoe

using namespace bitsmoe;

static bool quant_bits_ok(int bits) { return bits == 1 || bits == 2 || bits == 3 || bits == 4 || bits == 6 || bits == 8; }

extern "C" int bitsmoe_quantize_tiles(const float* rows, int64_t k, int64_t dim, int64_t row_stride, int32_t bits,
                                      int32_t iters, int8_t* levels_out, float* scale_out, void* stream) {
    BITSMOE_REQUIRE(quant_bits_ok(bits), "Unsupported bit width: %d", bits);
    BITSMOE_REQUIRE(k >= 0 && dim >= 0 && row_stride >= dim && iters >= 1, "invalid shape");
    if (k == 0 || dim == 0) return BITSMOE_OK;
    BITSMOE_REQUIRE(rows && levels_out && scale_out, "null pointer");
    const int64_t n_tiles = (dim + N_TILE - 1) / N_TILE;
    BITSMOE_REQUIRE(n_tiles < ((int64_t)1 << 24), "too many columns");
    const int64_t units = k * n_tiles;
    const int64_t blocks = std::min<int64_t>((units + 15) / 16, 65535);
    hipLaunchKernelGGL(k_quantize_tiles, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, rows, k, dim, row_stride,
                       (int)n_tiles, bits, iters, 1e-8f, levels_out, scale_out);
    BITSMOE_HIP_TRY(hipGetLastError());
    return BITSMOE_OK;
}

extern "C" int bitsmoe_pack_slabs(const int8_t* levels, const float* scale, int64_t k, int64_t dim, int32_t bits,
                                  uint32_t* payload_out, void* scale_out_f16, void* stream) {
    BITSMOE_REQUIRE(quant_bits_ok(bits), "Unsupported bit width: %d", bits);
    BITSMOE_REQUIRE(k >= 0 && dim >= 0, "invalid shape");
    if (k == 0 || dim == 0) return BITSMOE_OK;
    BITSMOE_REQUIRE(levels && scale && payload_out && scale_out_f16, "null pointer");
    const int64_t n_tiles = (dim + N_TILE - 1) / N_TILE;
    BITSMOE_REQUIRE(n_tiles < ((int64_t)1 << 24), "too many columns");
    const int64_t units = k * n_tiles * 2;
    const int64_t blocks = std::min<int64_t>((units + 3) / 4, 65535);
    hipLaunchKernelGGL(k_pack_slabs, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, levels, scale, k, (int)n_tiles,
                       bits, payload_out, (__half*)scale_out_f16);
    BITSMOE_HIP_TRY(hipGetLastError());
    return BITSMOE_OK;
}

extern "C" int bitsmoe_pack_matrix(const float* matrix, int64_t rank, int64_t dim, int64_t row_stride, const void* s_vec,
                                   int32_t s_is_f32, int32_t n_ranges, const int32_t* ranges, int32_t iters,
                                   uint32_t* payload_out, void* scale_out_f16, void* s_out_f16, int32_t* rank_idx_out,
                                   int32_t* tile_meta_out, int32_t* slab_meta_out, void* stream) {
    BITSMOE_REQUIRE(rank >= 0 && rank < ((int64_t)1 << 31) && dim > 0 && row_stride >= dim && iters >= 1 && n_ranges >= 0,
                    "invalid shape");
    if (n_ranges == 0) return BITSMOE_OK;
    BITSMOE_REQUIRE(matrix && ranges && payload_out && scale_out_f16, "null pointer");
    const bool tables = slab_meta_out != nullptr;
    BITSMOE_REQUIRE(!tables || (s_vec && s_out_f16 && rank_idx_out && tile_meta_out), "null pointer");
    const int64_t n_tiles = (dim + N_TILE - 1) / N_TILE;
    BITSMOE_REQUIRE(n_tiles < ((int64_t)1 << 24), "too many columns");
    PackTables tab = {};
    int64_t row = 0, pay = 0, sc = 0, slab = 0;
    for (int i = 0; i < n_ranges; ++i) {
        const int bits = ranges[3 * i], from = ranges[3 * i + 1], to = ranges[3 * i + 2];
        BITSMOE_REQUIRE(bits_supported(bits), "Unsupported bit width: %d", bits);
        BITSMOE_REQUIRE(0 <= from && from < to && to <= rank, "Invalid segment range (s=%d, e=%d) for rank=%lld", from, to,
                        (long long)rank);
        if (i == 0 || bits != ranges[3 * (i - 1)]) {
            if (tab.n_buckets) {
                const PackBucket& b = tab.bucket[tab.n_buckets - 1];
                pay += (int64_t)b.rows * MICROS * words_per_row(b.bits) * n_tiles;
                sc += (int64_t)b.rows * n_tiles;
                slab += (b.rows + K_SLAB - 1) / K_SLAB;
            }
            BITSMOE_REQUIRE(tab.n_buckets < PACK_MAX_BUCKETS, "rows of one width must be neighbouring ranges");
            tab.bucket[tab.n_buckets++] = PackBucket{pay, sc, bits, (int32_t)row, 0, (int32_t)slab};
        }
        tab.bucket[tab.n_buckets - 1].rows += to - from;
        row += to - from;
        BITSMOE_REQUIRE(row < ((int64_t)1 << 31), "too many rows");
    }
    const PackBucket& last = tab.bucket[tab.n_buckets - 1];
    pay += (int64_t)last.rows * MICROS * words_per_row(last.bits) * n_tiles;
    slab += (last.rows + K_SLAB - 1) / K_SLAB;
    tab.n_slabs = (int32_t)slab;
    BITSMOE_REQUIRE(!tables || (pay < ((int64_t)1 << 31) && slab * n_tiles < ((int64_t)1 << 31)),
                    "the tables' 32-bit offsets do not reach over %lld payload words", (long long)pay);
    // (a launch carries PACK_MAX_RANGES ranges by value; more of them take more launches)
    int32_t at = 0;      // packed rows so far, and the bucket of the range before
    int bucket = -1;
    for (int r0 = 0; r0 < n_ranges; r0 += PACK_MAX_RANGES) {
        tab.n_ranges = std::min(n_ranges - r0, PACK_MAX_RANGES);
        for (int k = 0; k < tab.n_ranges; ++k) {
            const int32_t* rg = ranges + 3 * (int64_t)(r0 + k);
            if (r0 + k == 0 || rg[0] != rg[-3]) ++bucket;
            tab.range[k] = PackRange{at, rg[1], bucket};
            at += rg[2] - rg[1];
        }
        tab.row_end = at;
        const bool first = r0 == 0;
        const int64_t rows_here = tab.row_end - tab.range[0].first;
        const int64_t unit_blocks = std::min<int64_t>((rows_here * n_tiles + 15) / 16, 1 << 20);
        const int64_t table_threads = tables ? rows_here + (first ? slab * n_tiles : 0) : 0;
        auto kernel = s_is_f32 ? k_pack_matrix<4> : k_pack_matrix<2>;
        hipLaunchKernelGGL(kernel, dim3((unsigned)(unit_blocks + (table_threads + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                           matrix, row_stride, dim, (int)n_tiles, s_vec, tab, iters, 1e-8f, (int)unit_blocks, payload_out,
                           (__half*)scale_out_f16, (__half*)s_out_f16, rank_idx_out, tile_meta_out, first ? slab_meta_out : nullptr);
        BITSMOE_HIP_TRY(hipGetLastError());
    }
    return BITSMOE_OK;
}
