// split.hpp -- f32 values as exact sums of bf16 parts (gfx950).
//
// The 16-bit matrix cores run 16 times the rate of the f32 ones.  An f32 value is the sum
// of three bf16 parts, each what is left rounded to nearest even (8 significant bits and a
// sign each: all 24 bits).  Rounded parts reach 2^-8 and 2^-16 of the value, with either
// sign, so the six products of parts down to that size hold a product to 0.9 * 2^-24, also
// with either sign (parts cut off instead reach twice and four times as far and shrink
// every product: 7.8 * 2^-24 at most).  A value that rounds up to infinity, or is one,
// leaves NaN in the lower parts.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace unillm {

typedef float split_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 split_bf16x2 __attribute__((ext_vector_type(2)));

// two f32 -> bf16 rounded to nearest even, packed, a in the low half
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t,
                              __builtin_convertvector(split_f32x2{a, b}, split_bf16x2));
}
__device__ __forceinline__ float bf16_lo(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t p) { return __uint_as_float(p & 0xFFFF0000u); }

// two f32 (as bits) -> their three bf16 parts, packed
__device__ __forceinline__ void split2(uint32_t a, uint32_t b, uint32_t& p0, uint32_t& p1,
                                       uint32_t& p2) {
    const float fa = __uint_as_float(a), fb = __uint_as_float(b);
    p0 = pack_bf16(fa, fb);
    const float a1 = fa - bf16_lo(p0), b1 = fb - bf16_hi(p0);
    p1 = pack_bf16(a1, b1);
    p2 = pack_bf16(a1 - bf16_lo(p1), b1 - bf16_hi(p1));
}

}  // namespace unillm
