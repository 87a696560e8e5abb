// fp32 values as sums of bf16 values, for products of fp32 operands on the 16-bit matrix cores.
//
// x = x1 + x2 + x3 with x1 = bf16(x), x2 = bf16(x - x1), x3 = bf16(x - x1 - x2), each rounded to nearest: the differences are exact,
// |x2| <= 2^-8 |x|, |x3| <= 2^-17 |x|, and what is left is below 2^-26 |x| (nothing, for nearly all x).  Of the nine products of
// two such sums six are kept, x1 y1, x1 y2, x2 y1, x1 y3, x2 y2, x3 y1; the others are at most 2^-24 |x y| together, of either sign, which
// is the size of one rounding of an fp32 product, and the six are exact and added up in fp32.
#pragma once
#include "common.h"

namespace pdw {

typedef __bf16 split_bf8 __attribute__((ext_vector_type(8)));
typedef float split_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t split_pack(float x, float y) {   // v_cvt_pk_bf16_f32
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{x, y}, b2));
}
__device__ __forceinline__ float split_lo(uint32_t p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float split_hi(uint32_t p) { return __builtin_bit_cast(float, p & 0xffff0000u); }

// The parts of two values, x in the low halves.
__device__ __forceinline__ void split_pair(float x, float y, uint32_t (&p)[3]) {
    p[0] = split_pack(x, y);
    const float rx = x - split_lo(p[0]), ry = y - split_hi(p[0]);
    p[1] = split_pack(rx, ry);
    p[2] = split_pack(rx - split_lo(p[1]), ry - split_hi(p[1]));
}

// Stays finite while the parts stand for the values: the third is NaN for an infinity, a NaN and a value that rounds up to infinity.
__device__ __forceinline__ float split_watch(const uint32_t (&p)[3], float seen) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    const b2 v = __builtin_bit_cast(b2, p[2]);
    return __builtin_amdgcn_fdot2_f32_bf16(v, v, seen, false);
}
__device__ __forceinline__ bool split_failed(float seen) { return !(seen < __builtin_inff()); }

}  // namespace pdw
