// fp32 products on the f16 matrix cores, at the accuracy of an fp32 kernel.
//
// hi = f16(x), lo = f16(x - hi), both rounded to nearest: 2 x 11 significant bits and the sign of lo hold 23 to 24 bits of x, all of them
// for three numbers in four and all but the last for the fourth.  A product is the sum of hi*hi, hi*lo and lo*hi; lo*lo, up to 2^-22 of it, is left out.  That is
// three matrix instructions per 16 values of k where three bf16 parts (bf16x3.hpp) take six, and 4 bytes an operand instead of 6.
// What it loses in the operands, 2^-24 of a product at random, it gains back in the accumulator, which is rounded once per matrix instruction:
// from 64 values of k on sums are no less exact than those of three bf16 parts (Winograd F(2x2,3x3) on normally distributed filters
// and rectified samples, rms against 64 bits, fp32 / three parts / two: 64 channels 2.3 / 1.7 / 1.7e-7, 256 channels 4.3 / 2.8 / 2.3e-7, 512 channels 5.9 / 3.8 / 3.0e-7).
// At random: where all products of a sum lose the same bits, nothing evens that out, and single maps and filters come out less exact than in three parts, which lose
// next to nothing of an operand.  Of 24 constants drawn for each (10 with 256 channels), rms of two parts next to three on average and at most, and next to fp32 at most: a flat map under
// normally distributed filters 0.92, 1.47, 1.35 with 64 channels and 0.83, 1.07, 0.75 with 256; channels flat in themselves 1.00, 1.52, 0.90 and 0.82, 1.07,
// 0.63; a flat map under one box filter, where three parts reach 0.1 to 0.8e-7 and fp32 5 to 14e-7, 1.72, 4.16, 0.43 and 1.32, 4.27, 0.55.  A caller who wants the
// bits that such data leaves has them with DR_WINO_PAIR=0.
//
// f16 ends at 65504 and 2^-24, which the operands have to be scaled for: with the largest between 2^11 and 2^15, what smaller ones lose is below
// 2^-36 of the largest.  f16 denormals are multiplied like other numbers.
#pragma once

#include "bf16x3.hpp"

namespace drhip {

typedef _Float16 f16x2h __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8h __attribute__((ext_vector_type(8)));

__device__ inline unsigned pack_f16(float a, float b) { return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2b{a, b}, f16x2h)); }
// minusOne: -1, from where the compiler does not see it; then the conversion of hi and the difference are one instruction.
__device__ inline float f16_rest(float x, unsigned packed, int which, float minusOne) {
    return fmaf((float)__builtin_bit_cast(f16x2h, packed)[which], minusOne, x);
}

__device__ inline f32x16b mfma_f16(u32x4b a, u32x4b b, f32x16b c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8h, a), __builtin_bit_cast(f16x8h, b), c, 0, 0, 0);
}

}  // namespace drhip
