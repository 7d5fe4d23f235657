// gemm_split.hpp -- fp32 products on the bf16 matrix units.
//
// gfx950's bf16 MFMA does 16 times the fp32 MFMA's work per cycle, so an
// fp32 product is taken there as a sum of bf16 ones, without giving up fp32's
// precision:
//   * Each fp32 value x is cut into three bf16 values h + m + l = x exactly:
//     h = bf16(x), m = bf16(x - h), l = x - h - m, each rounded to nearest.
//     8 bits each and a sign hold all 24 bits, and both differences are exact.
//   * a·b is the sum of six of the nine bf16 products: h·h, and h·m, m·h, m·m,
//     h·l, l·h, which are 2^-8 of it and less.  |m| <= 2^-8 |x| and |l| <= 2^-17
//     |x|, so the three left out (m·l, l·m, l·l) come to at most 2^-24 of a·b,
//     as much as one rounding of the fp32 sum.  That is reached where both
//     operands sit just below half an ulp of bf16 (0x1.00ff8p+0, 2^-24.01), and
//     a sum of such products of one sign is off by as much; normal values: rms
//     2^-27.4, 3 % of the products beyond 2^-26, either sign (a sum of one or two
//     products is no better than fp32's, longer ones are).
//   * Every bf16 product is exact in fp32, and the matrix unit accumulates in
//     fp32.  h·h has an accumulator of its own, and the five small products
//     share a second one: the large sum is then rounded once per instruction
//     (16 products of k; the fp32 instruction takes two) and the roundings of
//     the small sum weigh 2^-8.  In one accumulator the unit's rounding, which
//     is not to nearest, showed: sums of 10^5 terms came out 4e-6 of their rms
//     low.  The two are added at the end.
// Measured against 64 bits (2-norm, fp32 MFMA / this), normal values: K = 16:
// 7.5e-8 / 3.2e-8, 256: 2.9e-7 / 8.9e-8, 4096: 1.14e-6 / 3.9e-7, 16384: 2.3e-6 /
// 8.2e-7, 100352: 5.7e-6 / 2.0e-6; sums of one sign, K = 256: 1.7e-7 / 7.9e-8,
// 4096: 7.0e-7 / 3.5e-7; half the values zero, K = 2304: 6.1e-7 / 2.3e-7.
//
// Range: l reaches 2^-24 below x, and bf16 has fp32's exponents, so the parts
// of an x below 2^-102 would drop bits.  The operands are therefore scaled by
// 2^24 before the cut and the sums by 2^-48 at the end (both exact); then every
// fp32 value, subnormal ones too, keeps all its bits.  What the scaling puts
// out of range instead -- values above 2^103, sums above 2^80 -- and every
// infinity or NaN among the operands comes out as an infinity or a NaN here
// (split_finish): the workgroup then takes its tile again with fp32 MFMAs, so
// such operands give what they always gave.
//
// Cost: a bf16 MFMA of 32x32x16 takes 32 cycles of its SIMD's matrix unit, so
// six of them take 192 where the fp32 ones took 512, and about four vector
// instructions run beside each (two waves per SIMD: 34, 37, 44, 51 cycles per
// MFMA with 0, 4, 6, 8 of them; beside an fp32 MFMA none do).
// v_dot2_f32_bf16, which would take a part out and subtract it in one, does not
// (59 cycles with two), hence the shifts.
#pragma once

#include "gemm_kernel.hpp"

namespace mtk {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kSplitScale = 0x1p24f;
constexpr float kSplitUnscale = 0x1p-48f;

// Two floats to a bf16 pair, rounded to nearest (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
    const bf16x2 r = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ float bf16_lo(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }

// The parts h, m, l of four values.
__device__ __forceinline__ void split4(const f32x4& x, u32x2& h, u32x2& m, u32x2& l) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float x0 = x[2 * i] * kSplitScale, x1 = x[2 * i + 1] * kSplitScale;
        h[i] = bf16_pair(x0, x1);
        const float r0 = x0 - bf16_lo(h[i]), r1 = x1 - bf16_hi(h[i]);
        m[i] = bf16_pair(r0, r1);
        l[i] = bf16_pair(r0 - bf16_lo(m[i]), r1 - bf16_hi(m[i]));
    }
}

// The parts of the eight k-values that one lane gives to an MFMA (lane l: row
// l%32 of a 32-row block, the k of half l/32 of a 16-deep chunk).
struct SplitFrag {
    u32x4 h, m, l;
};

// (B's fragment first: the accumulator holds the transposed block, as
// mfma_32x32x2.)
__device__ __forceinline__ f32x16 mfma_bf16(const u32x4& a, const u32x4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, b),
                                                   __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
}

// Products P0..P1-1 (of six) of one 16-deep chunk: acc + sml += A·B at the scale
// of 2^48; consecutive MFMAs feed different accumulators.
template <int MB, int NB, int P0, int P1>
__device__ __forceinline__ void mfma_split(f32x16 (&acc)[MB][NB], f32x16 (&sml)[MB][NB],
                                           const SplitFrag (&a)[MB], const SplitFrag (&b)[NB]) {
#pragma unroll
    for (int p = P0; p < P1; ++p)
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                f32x16& c = p == 0 ? acc[i][j] : sml[i][j];
                c = mfma_bf16((p == 2 || p == 3) ? a[i].m : p == 4 ? a[i].l : a[i].h,
                              (p == 1 || p == 3) ? b[j].m : p == 5 ? b[j].l : b[j].h, c);
            }
}

template <int MB, int NB>
__device__ __forceinline__ void zero_blocks(f32x16 (&acc)[MB][NB]) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
}

// acc = the two sums together, without the scale; true where one of them is an
// infinity or a NaN.
template <int MB, int NB>
__device__ __forceinline__ bool split_finish(f32x16 (&acc)[MB][NB], const f32x16 (&sml)[MB][NB]) {
    float z = 0.f;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] = (acc[i][j][r] + sml[i][j][r]) * kSplitUnscale;
                z = __builtin_fmaf(acc[i][j][r], 0.f, z);
            }
    return z != z;
}

}  // namespace mtk
