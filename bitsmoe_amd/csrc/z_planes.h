// z = silu(gate) * up as an operand of the block-scaled 16x16x128 MFMA (v_mfma_scale_f32_16x16x128_f8f6f4), whose other
// operand is the packed codes of a down matrix AS THEY ARE.
//
// A code of up to two bits in a nibble IS an fp4 (E2M1) number, code / 2; a code of up to four bits in a 6-bit field IS an fp6
// (E2M3) number, code / 8.  So the 2-bit payload needs one mask (and, for every other register, one shift) per EIGHT weights,
// where an f16 operand needs a rotate and an and-or per two, and no 16-bit rounding of weights.  z goes in as three fp6 planes:
//
//     z = scale * (p0 + 2^-5 p1 + 2^-10 p2),   scale = 2^(e - 1), e the exponent of the largest |z| of 32 neighbouring columns
//
// p0 = z / scale rounded to E2M3 (|p0| <= 4, three fraction bits: a remainder of at most 1/8), p1 and p2 the remainders of the
// plane before it, 32 times as large (at most 4 again).  What is left is at most 2^-14 of the block's largest |z|.  The planes
// are made of the fp32 product (as an f16 number and the f16 remainder): they take the place of z's rounding to f16, they do
// not come on top of it.  And the constant term of the codes is taken of the sum of the PLANES: of the sum of z, the planes' error
// would enter times the code instead of times the level.  Error of the operator against 64-bit sums (f16 / bf16, 512 to 1408
// columns, 1 to 900 tokens), against f16 operands: decode kernels 4.3e-4 .. 5.4e-4 -> 4.0e-4 .. 4.5e-4, grouped GEMM 5.1e-4 .. 5.9e-4 ->
// 4.7e-4 .. 5.5e-4.
// A block with an infinity or a NaN has the NaN scale: its products are NaN, as they are where the constant
// term of an f16 operand is subtracted.
//
// Rates on one MI355X, all CUs: 10.5 ns per fp4 x fp6 MFMA of 16x16x128 and SIMD, 7.9 per f16 16x16x32, i.e. three planes
// cost what the f16 form's four k-steps cost (31.4 and 31.8 ns); the gain is what stands beside the MFMAs.  Down kernels under
// the tracer, f16 operands -> planes: 64 tokens on 128 experts 26.4 -> 24.5 us, 256 tokens on 512 experts 54.9 -> 50.9, 23 tokens on 64
// checkpoint-shaped experts 13.6 -> 12.3; grouped GEMM 333 tokens on 64 experts 42.0 -> 32.5, 4096 tokens on 128 experts 146 -> 129 (its
// SiLU pass, which makes the planes, 25.6 -> 31).
//
// The record of 32 columns is 20 words: p0 (6), p1 (6), p2 (6), the three scale bytes (E8M0, byte p for plane p), and the sum of
// the planes over the record's whole TILE of 128 columns where the grouped GEMM wants it.  It is kept as five 16-byte pieces.
#pragma once

#include "fast_helpers.h"

namespace bitsmoe {

typedef _Float16 f16x32 __attribute__((ext_vector_type(32)));
typedef uint32_t u32x6 __attribute__((ext_vector_type(6)));
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

constexpr int ZR_PIECES = 5;       // 16-byte pieces of a record
constexpr int Z_BLOCK = 32;        // columns of a record
constexpr int ZB_BYTES = ZR_PIECES * 64 * 16;      // the records of 16 rows x 128 columns
constexpr int Z_FMT_FP6 = 2, Z_FMT_FP4 = 4;      // operand formats of the MFMA

// E8M0 scales (four equal bytes) that undo a format's unit: codes of the low fp4 plane, of the high one (4 times), of fp6
constexpr int W_SCALE_FP4 = 0x80808080, W_SCALE_FP4_HI = 0x82828282;
constexpr int W_SCALE_FP6 = 0x82828282;

__device__ __forceinline__ uint32_t pk_sub_f16(uint32_t a, uint32_t b) {
    const h2 r = __builtin_bit_cast(h2, a) - __builtin_bit_cast(h2, b);
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

// v of the four lanes of a quad, added up (every lane gets the sum)
__device__ __forceinline__ float quad_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));      // lanes 1, 0, 3, 2
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true));      // lanes 2, 3, 0, 1
    return v;
}

// A record's pieces, and 32 f16 values (a: the first eight).  (Members, no arrays: the compiler keeps arrays of vectors that are
// written in one unrolled loop and read in another in scratch memory.)
struct ZRecord {
    u32x4 a, b, c, d, e;
};
struct F16x32 {
    u32x4 a, b, c, d;
};

__device__ __forceinline__ u32x16 regs_of(const F16x32& v) {
    return __builtin_shufflevector(__builtin_shufflevector(v.a, v.b, 0, 1, 2, 3, 4, 5, 6, 7),
                                   __builtin_shufflevector(v.c, v.d, 0, 1, 2, 3, 4, 5, 6, 7), 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13,
                                   14, 15);
}
__device__ __forceinline__ float sum_f16(u32x16 v, float s) {
    typedef __fp16 h2v __attribute__((ext_vector_type(2)));
    const h2v ones = {(__fp16)1.0f, (__fp16)1.0f};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const uint32_t w = v[i];
        s = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2v, w), ones, s, false);
    }
    return s;
}

// silu(g) * u of two neighbouring columns: z_operand's f16 values and the f16 remainders of the fp32 products
struct ZPair {
    uint32_t hi, lo;
};
__device__ __forceinline__ ZPair z_pair(float g0, float u0, float g1, float u1) {
    float p0 = silu_f32(g0) * u0, p1 = silu_f32(g1) * u1;
    asm("" : "+v"(p0));      // (a value of its own: z_operand)
    asm("" : "+v"(p1));
    ZPair r;
    r.hi = f16_pair(p0, p1);
    const h2 h = __builtin_bit_cast(h2, r.hi);
    r.lo = f16_pair(p0 - (float)h[0], p1 - (float)h[1]);
    return r;
}

// The record of 32 values hi + lo (f16 numbers and their remainders).  SUM: `sum` receives the sum of the planes (the record's last
// word is left to the caller).
template <bool SUM>
__device__ __forceinline__ ZRecord z_record(const F16x32& hi, const F16x32& lo, float& sum) {
    u32x16 v = regs_of(hi);
    uint32_t top = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) top = pk_max_u16(top, v[i] & 0x7FFF7FFFu);
    const uint32_t e16 = max(top & 0xFFFFu, top >> 16) >> 10;       // the largest exponent field (0: subnormals)
    const uint32_t e8 = max(e16, 1u) + 111u;                        // E8M0 of 2^(e - 1)
    const float s0 = __uint_as_float(e8 << 23), s1 = __uint_as_float((e8 - 5u) << 23), s2 = __uint_as_float((e8 - 10u) << 23);
    // (the remainders of an f16 number are exact; pair by pair, or the compiler subtracts the 32 values one by one)
    auto to_fp6 = [&](float s) { return __builtin_amdgcn_cvt_scalef32_pk32_fp6_f16(__builtin_bit_cast(f16x32, v), s); };
    auto value = [](u32x6 p, float s) { return __builtin_bit_cast(u32x16, __builtin_amdgcn_cvt_scalef32_pk32_f16_fp6(p, s)); };
    if constexpr (SUM) sum = 0.0f;
    const u32x6 p0 = to_fp6(s0);
    {
        const u32x16 b = value(p0, s0), l = regs_of(lo);
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = pk_add_f16(pk_sub_f16(v[i], b[i]), l[i]);
        if constexpr (SUM) sum = sum_f16(b, sum);
    }
    const u32x6 p1 = to_fp6(s1);
    {
        const u32x16 b = value(p1, s1);
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = pk_sub_f16(v[i], b[i]);
        if constexpr (SUM) sum = sum_f16(b, sum);
    }
    const u32x6 p2 = to_fp6(s2);
    if constexpr (SUM) sum = sum_f16(value(p2, s2), sum);
    ZRecord r;
    r.a = u32x4{p0[0], p0[1], p0[2], p0[3]};
    r.b = u32x4{p0[4], p0[5], p1[0], p1[1]};
    r.c = u32x4{p1[2], p1[3], p1[4], p1[5]};
    r.d = u32x4{p2[0], p2[1], p2[2], p2[3]};
    r.e = u32x4{p2[4], p2[5], e16 == 31u ? 0x00FFFFFFu : e8 * 0x010101u - 0x0A0500u, 0u};
    return r;
}

// z as 32 f16 values from its record
__device__ __forceinline__ F16x32 z_from_record(const ZRecord& r) {
    const u32x6 p0 = {r.a[0], r.a[1], r.a[2], r.a[3], r.b[0], r.b[1]};
    const u32x6 p1 = {r.b[2], r.b[3], r.c[0], r.c[1], r.c[2], r.c[3]};
    const u32x6 p2 = {r.d[0], r.d[1], r.d[2], r.d[3], r.e[0], r.e[1]};
    const uint32_t e8 = r.e[2] & 0xFFu;
    const float s0 = __uint_as_float(e8 == 255u ? 0x7FC00000u : e8 << 23);
    const float s1 = s0 * 0x1p-5f, s2 = s0 * 0x1p-10f;
    // (the small planes first)
    auto plane = [](u32x6 p, float s) { return __builtin_bit_cast(u32x16, __builtin_amdgcn_cvt_scalef32_pk32_f16_fp6(p, s)); };
    const u32x16 v2 = plane(p2, s2), v1 = plane(p1, s1), v0 = plane(p0, s0);
    u32x16 v;
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = pk_add_f16(v0[i], pk_add_f16(v1[i], v2[i]));
    return F16x32{u32x4{v[0], v[1], v[2], v[3]}, u32x4{v[4], v[5], v[6], v[7]}, u32x4{v[8], v[9], v[10], v[11]},
                  u32x4{v[12], v[13], v[14], v[15]}};
}

// ---- the operands of one 16-row block x 128 columns
struct ZOperand {
    i32x8 p[3];      // (an fp6 operand is the first six words)
    int scales;
};
__device__ __forceinline__ ZOperand z_operand_of(const ZRecord& r) {
    const u32x4 a = opaque(r.a), b = opaque(r.b), c = opaque(r.c), d = opaque(r.d), e = opaque(r.e);
    ZOperand o;
    o.p[0] = i32x8{(int)a[0], (int)a[1], (int)a[2], (int)a[3], (int)b[0], (int)b[1], 0, 0};
    o.p[1] = i32x8{(int)b[2], (int)b[3], (int)c[0], (int)c[1], (int)c[2], (int)c[3], 0, 0};
    o.p[2] = i32x8{(int)d[0], (int)d[1], (int)d[2], (int)d[3], (int)e[0], (int)e[1], 0, 0};
    o.scales = (int)e[2];
    return o;
}

// The codes of row block nb of a block (wave_layout.h, role 1) as MFMA operands: 2-bit one fp4 operand, 3-bit one fp6 operand,
// 4-bit two fp4 operands (the low and the high two bits).
template <int W, int NB>
__device__ __forceinline__ void code_operands(u32x4 q0, u32x4 q1, u32x4 q2, u32x4 q3, i32x8& op, i32x8& op_hi) {
    constexpr uint32_t M4 = 0x33333333u;
    if constexpr (W == 2) {
        const uint32_t x = block_word<2 * NB>(q0, q1, q2, q3), y = block_word<2 * NB + 1>(q0, q1, q2, q3);
        op = i32x8{(int)(x & M4), (int)((x >> 2) & M4), (int)(y & M4), (int)((y >> 2) & M4), 0, 0, 0, 0};
    } else if constexpr (W == 4) {
        const uint32_t w0 = block_word<4 * NB>(q0, q1, q2, q3), w1 = block_word<4 * NB + 1>(q0, q1, q2, q3), w2 = block_word<4 * NB + 2>(q0, q1, q2, q3), w3 = block_word<4 * NB + 3>(q0, q1, q2, q3);
        op = i32x8{(int)(w0 & M4), (int)(w1 & M4), (int)(w2 & M4), (int)(w3 & M4), 0, 0, 0, 0};
        op_hi = i32x8{(int)((w0 >> 2) & M4), (int)((w1 >> 2) & M4), (int)((w2 >> 2) & M4), (int)((w3 >> 2) & M4), 0, 0, 0, 0};
    } else {
        // low three bits of every 6-bit field of the pair's 192 bits (even row block), or the high three (odd)
        constexpr int G = 6 * (NB >> 1);
        constexpr uint32_t M0 = 0xC71C71C7u, M1 = 0x71C71C71u, M2 = 0x1C71C71Cu;
        const uint32_t w0 = block_word<G>(q0, q1, q2, q3), w1 = block_word<G + 1>(q0, q1, q2, q3), w2 = block_word<G + 2>(q0, q1, q2, q3), w3 = block_word<G + 3>(q0, q1, q2, q3), w4 = block_word<G + 4>(q0, q1, q2, q3),
                       w5 = block_word<G + 5>(q0, q1, q2, q3);
        if constexpr ((NB & 1) == 0) {
            op = i32x8{(int)(w0 & M0), (int)(w1 & M1), (int)(w2 & M2), (int)(w3 & M0), (int)(w4 & M1), (int)(w5 & M2), 0, 0};
        } else {
            auto sh = [](uint32_t hi, uint32_t lo) { return __builtin_amdgcn_alignbit(hi, lo, 3u); };
            op = i32x8{(int)(sh(w1, w0) & M0), (int)(sh(w2, w1) & M1), (int)(sh(w3, w2) & M2),
                       (int)(sh(w4, w3) & M0), (int)(sh(w5, w4) & M1), (int)((w5 >> 3) & M2), 0, 0};
        }
    }
}

// The operand that makes minus the sum of the other one: -1 in every place (fp4), times 2^(W-1) by its scale.
__device__ __forceinline__ i32x8 minus_ones() {
    constexpr int V = (int)0xAAAAAAAAu;
    return i32x8{V, V, V, V, 0, 0, 0, 0};
}
constexpr int minus_ones_scale(int w) { return 0x01010101 * (127 + w - 1); }

template <int W>
struct CodeFormat {
    static constexpr int FMT = W == 3 ? Z_FMT_FP6 : Z_FMT_FP4;
    static constexpr int SCALE = W == 3 ? W_SCALE_FP6 : W_SCALE_FP4;
};

// t += z (rows: assignments) x codes (columns: output rows), plane P; CODES_FIRST: the two change places
template <int FMT, int P, bool CODES_FIRST>
__device__ __forceinline__ f32x4 mfma_plane(const ZOperand& z, const i32x8& codes, int code_scale, f32x4 t) {
    if constexpr (CODES_FIRST)
        return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(codes, z.p[P], t, FMT, Z_FMT_FP6, 0, code_scale, P, z.scales);
    else
        return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(z.p[P], codes, t, Z_FMT_FP6, FMT, P, z.scales, 0, code_scale);
}

}  // namespace bitsmoe
