// split.hpp -- f32 values as exact sums of bf16 parts (gfx950).
//
// The 16-bit matrix cores run 16 times the rate of the f32 ones.  An f32 value split by
// truncation into three bf16 parts (8 significant bits each) keeps all its 24 bits, and
// the six products of parts down to 2^-16 of the leading one hold an f32 product to
// 2^-24: f32 matrix products at 16 / 6 of the f32 rate.  Truncation cannot overflow; an
// infinity keeps its kind in part 0 and makes the lower parts NaN.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace unillm {

typedef uint32_t split_u32x4 __attribute__((ext_vector_type(4)));

// two f32 (as bits) -> their upper halves packed, lo in the low half
__device__ __forceinline__ uint32_t pack_hi(uint32_t lo, uint32_t hi) {
    return __builtin_amdgcn_perm(hi, lo, 0x07060302u);
}

// two f32 (as bits) -> their three bf16 parts, packed
__device__ __forceinline__ void split2(uint32_t a, uint32_t b, uint32_t& p0, uint32_t& p1,
                                       uint32_t& p2) {
    p0 = pack_hi(a, b);
    const float a1 = __uint_as_float(a) - __uint_as_float(a & 0xFFFF0000u);
    const float b1 = __uint_as_float(b) - __uint_as_float(b & 0xFFFF0000u);
    const uint32_t ua = __float_as_uint(a1), ub = __float_as_uint(b1);
    p1 = pack_hi(ua, ub);
    const float a2 = a1 - __uint_as_float(ua & 0xFFFF0000u);
    const float b2 = b1 - __uint_as_float(ub & 0xFFFF0000u);
    p2 = pack_hi(__float_as_uint(a2), __float_as_uint(b2));
}

}  // namespace unillm
