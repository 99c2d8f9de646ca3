// fp32 products on the bf16 matrix cores, at fp32 accuracy.
//
// An fp32 number is the sum of three bf16 numbers: hi = bf16(x), mid = bf16(x - hi), lo = bf16(x - hi - mid), each
// rounded to nearest.  The differences are exact, and 3 x 8 significant bits (with the signs of the parts) hold all 24
// of x, so nothing of the operand is lost.  A product is then the sum of nine partial products, each exact in fp32;
// the three that are left out (mid*lo, lo*mid, lo*lo) are below 2^-26 of the product, less than the rounding of a
// single fp32 multiplication.  The other six go to v_mfma_f32_32x32x16_bf16, which accumulates in fp32: six matrix
// instructions of 32 clocks for 16 values of k against eight of 64 clocks on the fp32 matrix path - 2.67 times the
// rate - and one rounding of the accumulator per instruction instead of one per product.  (Measured, 32x16 by
// 16x32 with operands in [-0.5, 0.5): 3.3e-8 relative against 7.3e-8 for a chain of fp32 FMAs; 2.34 PFLOP/s of matrix
// instructions sustained, and up to six vector instructions per matrix instruction ride along for nothing, where
// an fp32 MFMA and a vector instruction exclude each other.)
//
// bf16 ends at 2^-133, so that below 2^-110 the third part would lose bits that fp32 has.  Both operands are therefore multiplied by
// 2^16 when they are split, which puts the last bit of the smallest fp32 number there, and results by 2^-32.  What that takes
// out of range at the other end (operands above 2^111, results above 2^95) comes out as infinity or NaN, which the kernels that
// use this look for and work out again in fp32.
#pragma once

#include "drhip_common.hpp"

namespace drhip {

typedef float f32x16b __attribute__((ext_vector_type(16)));
typedef float f32x2b __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4b __attribute__((ext_vector_type(4)));
typedef unsigned u32x2b __attribute__((ext_vector_type(2)));

constexpr float kSplitScale = 0x1p16f, kSplitUnscaleOne = 0x1p-16f, kSplitUnscale = 0x1p-32f;

struct Bf16Pair3 { unsigned hi, mid, lo; };         // two values, each as three parts, packed by part

// 11 vector instructions for two values.  (v_dot2_f32_bf16 would take a residual in one instruction instead of two, but
// it runs on the matrix pipe: 8 clocks that no MFMA can use.)
__device__ inline Bf16Pair3 split_pair(float a, float b) {
    Bf16Pair3 p;
    p.hi = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2b{a, b}, bf16x2));
    const float ra = a - __builtin_bit_cast(float, p.hi << 16), rb = b - __builtin_bit_cast(float, p.hi & 0xffff0000u);
    p.mid = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2b{ra, rb}, bf16x2));
    const float sa = ra - __builtin_bit_cast(float, p.mid << 16), sb = rb - __builtin_bit_cast(float, p.mid & 0xffff0000u);
    p.lo = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2b{sa, sb}, bf16x2));
    return p;
}

__device__ inline f32x16b mfma_bf16(u32x4b a, u32x4b b, f32x16b c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The six partial products, smallest first: part of a, part of b (0 = hi, 1 = mid, 2 = lo).
constexpr int kProdA[6] = {2, 1, 0, 1, 0, 0};
constexpr int kProdB[6] = {0, 1, 2, 0, 1, 0};

// One element's parts as 16-bit patterns (filter banks, written once when a layer is prepared).  What has no parts, an infinity,
// a NaN or a value above 2^111, gets an infinite first part, so that nothing finite comes of it, and its own 32 bits as the others.
__device__ inline void split_one(float x, unsigned short (&part)[3]) {
    const unsigned bits = __float_as_uint(x);
    const bool fits = fabsf(x) < 0x1p111f;
    const Bf16Pair3 p = split_pair(fits ? kSplitScale * x : 0.0f, 0.0f);
    part[0] = (unsigned short)(fits ? p.hi : 0x7f80u);
    part[1] = (unsigned short)(fits ? p.mid : bits >> 16);
    part[2] = (unsigned short)(fits ? p.lo : bits);
}
__device__ inline float whole(unsigned hi, unsigned mid, unsigned lo) {
    if (hi == 0x7f80u) return __uint_as_float(mid << 16 | lo);
    return kSplitUnscaleOne * (__uint_as_float(lo << 16) + __uint_as_float(mid << 16) + __uint_as_float(hi << 16));
}

}  // namespace drhip
