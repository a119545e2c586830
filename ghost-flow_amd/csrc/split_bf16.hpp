// split_bf16.hpp -- an fp32 value as the sum of three bf16 pieces.
//
// x = p0 + p1 + p2 with p0 = bf16(x), p1 = bf16(x - p0), p2 = x - p0 - p1:
// each piece rounds to nearest and takes 8 significant bits, and both
// differences are exact in fp32, so the three carry all 24 bits of x down to
// 2^-133, the last bit of a bf16 subnormal (the bf16 matrix instructions keep
// subnormal operands and products).  fp32 goes on to 2^-149: a value scaled by
// kPieceUp before the split keeps all its bits whatever its size (from 2^112
// on its leading piece is infinite).  A product of two split values is taken as
//   a2 b0 + a1 b1 + a0 b2 + a1 b0 + a0 b1 + a0 b0
// -- every piece product exact in fp32, summed in the fp32 accumulator.  What
// is left out (a1 b2, a2 b1, a2 b2) is below 2^-24 of the product (a single
// product that stands alone in its sum is off by up to 0.93 ulp, rms 0.296,
// where one rounding gives 0.5 and 0.289).
#pragma once

#include "common.hpp"

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

namespace gfh {

constexpr float kPieceUp = 0x1p16f;     // before the split, of either operand
constexpr float kPieceDown = 0x1p-32f;  // for sums of products of two scaled operands

// The pieces of (x, y), packed with x in the low half.
__device__ __forceinline__ void split2(float x, float y, uint32_t &p0, uint32_t &p1, uint32_t &p2) {
#pragma clang fp contract(off)
    auto pack = [](float a, float b) __attribute__((always_inline)) {
        const f32x2 v = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
    };
    p0 = pack(x, y);
    const float x1 = x - __uint_as_float(p0 << 16), y1 = y - __uint_as_float(p0 & 0xffff0000u);
    p1 = pack(x1, y1);
    const float x2 = x1 - __uint_as_float(p1 << 16), y2 = y1 - __uint_as_float(p1 & 0xffff0000u);
    p2 = pack(x2, y2);
}

}  // namespace gfh
