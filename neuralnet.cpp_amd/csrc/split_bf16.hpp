// split_bf16.hpp — float32 products on the bf16 matrix cores, by exact splitting
// (three bf16 of a float32 and six of the nine part products: Henry, Tang and
// Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", ARITH 2019).
//
// A float x (scaled by 2^24) is the sum of three bf16 values, each the round
// to nearest of what the ones before it leave: h = bf16(x), m = bf16(x - h),
// l = bf16(x - h - m). A bf16 holds 8 significant bits, so three hold the 24
// of a float32. A product a b is then
//
//   ah bh + (ah bm + am bh) + (am bm + ah bl + al bh) + [am bl + al bm + al bl]
//
// where the bracket is at most (2^-24 + 2^-34) |a b| (|m| <= 2^-8 |x| and
// |l| <= 2^-17 |x|: half a unit in the last of 8 bits each; a = b = 1 + 2^-8 -
// 2^-17 comes within 1 % of it) and is left out: six bf16 products, exact in
// the matrix core's float32 accumulator, in place of one float32 product. So
// one product alone can be further off than the one rounding of a float32
// product, and sums of one or two products stay on the float32 cores; from
// three on the float32 chain's roundings weigh more. The bf16 matrix cores run
// 16 times the float32 ones' rate (measured on MI355X, independent streams:
// 2090 against 141 TFLOP/s), so six products still take 2.5 times less.
// ah bh goes to one accumulator and the five small ones to another: against
// 64-bit sums of normal inputs the error is 1.6e-7 at K 768 and 5.9e-7 at
// K 8192, the float32 matrix core's chain 4.6e-7 and 1.6e-6.
//
// The scale 2^24 keeps every part of every float32 input, denormals among
// them, a normal bf16 (no part is lost below 2^-126); results are scaled back
// by 2^-48. Inputs that reach 2^104 when rounded to bf16, results (or partial
// sums) from 2^80 on, infinities and NaN leave a value that is not finite: the
// caller checks for that and forms the output again on the float32 matrix
// cores. Below that the parts are exact: the remainder that split_part takes
// was compared with x - bf16(x) on MI355X, 8192 values of every exponent.
#pragma once

#include <hip/hip_runtime.h>

namespace nnhip
{

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

constexpr float kSplitScale = 0x1p24f;       // of each input
constexpr float kSplitUnscale = 0x1p-48f;    // of a product of two

// What rounding to bf16 leaves of two floats: x0 - bf16(x0) and x1 - bf16(x1),
// exact. One instruction each: the pair's dot product with (-1, 0) or (0, -1)
// added to x. The two constants are kept in scalar registers (the packed
// form of the inline constant -1 is not one of them).
struct SplitUnits
{
    bf16x2 e0, e1;
    __device__ __forceinline__ SplitUnits()
    {
        unsigned c0 = 0x0000bf80u, c1 = 0xbf800000u;
        asm("" : "+s"(c0));
        asm("" : "+s"(c1));
        e0 = __builtin_bit_cast(bf16x2, c0);
        e1 = __builtin_bit_cast(bf16x2, c1);
    }
};
__device__ __forceinline__ bf16x2 split_part(const SplitUnits& u, float& x0, float& x1)
{
    const bf16x2 p = __builtin_convertvector((floatx2){x0, x1}, bf16x2);
    x0 = __builtin_amdgcn_fdot2_f32_bf16(p, u.e0, x0, false);
    x1 = __builtin_amdgcn_fdot2_f32_bf16(p, u.e1, x1, false);
    return p;
}

// The three parts of eight floats that are scaled already.
__device__ __forceinline__ void split3_scaled(const SplitUnits& u, floatx8 x, bf16x8& h, bf16x8& m, bf16x8& l)
{
    uintx4 hv, mv, lv;
#pragma unroll
    for (int p = 0; p < 4; ++p)
    {
        float x0 = x[2 * p], x1 = x[2 * p + 1];
        hv[p] = __builtin_bit_cast(unsigned, split_part(u, x0, x1));
        mv[p] = __builtin_bit_cast(unsigned, split_part(u, x0, x1));
        lv[p] = __builtin_bit_cast(unsigned, __builtin_convertvector((floatx2){x0, x1}, bf16x2));
    }
    h = __builtin_bit_cast(bf16x8, hv);
    m = __builtin_bit_cast(bf16x8, mv);
    l = __builtin_bit_cast(bf16x8, lv);
}
// The three parts of eight floats.
__device__ __forceinline__ void split3(const SplitUnits& u, floatx8 x, bf16x8& h, bf16x8& m, bf16x8& l)
{
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] *= kSplitScale;
    split3_scaled(u, x, h, m, l);
}

// acc += the FM x FN blocks of 32 x 32 x 16 products' large parts, small += their five small ones; neighbouring
// instructions go to different accumulators.
template <int FM, int FN>
__device__ __forceinline__ void mfma_split(const bf16x8 (&a)[FM][3], const bf16x8 (&b)[FN][3],
                                           floatx16 (&acc)[FM][FN], floatx16 (&small)[FM][FN])
{
    constexpr int pa[6] = {0, 0, 2, 1, 0, 1}, pb[6] = {0, 2, 0, 1, 1, 0};
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
            {
                floatx16& c = t == 0 ? acc[i][j] : small[i][j];
                c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][pa[t]], b[j][pb[t]], c, 0, 0, 0);
            }
}

} // namespace nnhip
