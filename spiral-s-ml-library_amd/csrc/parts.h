// A f32 as the sum of three bf16 numbers, for products on the bf16 matrix pipe.
//
// Every f32 is the exact sum of three bf16 numbers, x = h + m + l: h is x rounded to bf16, m what is left rounded to bf16, l
// the rest (8 significant bits each and two signs: 24 bits and more).  A product of two f32 is then nine products of bf16, of
// which the three smallest (m l, l m, l l) are below 2^-24 of it, of either sign, and are left out.
#pragma once
#include "common.h"

namespace sp {

typedef __bf16 parts_bf16x2 __attribute__((ext_vector_type(2)));
typedef float parts_f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned parts_u32x4 __attribute__((ext_vector_type(4)));
typedef float parts_f32x4 __attribute__((ext_vector_type(4)));

// The range in which parts hold a number to the last bit: zero, and magnitudes from 2^-110 (the last bit of the lowest part is
// then no smaller than the smallest bf16, 2^-133; the pipe keeps subnormal numbers) up to where the bf16 is still finite.
// Tracked as the smallest non-zero 2 |x|, in bits and less one (zeros wrap to the largest).
constexpr unsigned PARTS_TINY = (127u - 110u) << 24;     // 2^-110 in that form, before the one is taken off
__device__ __forceinline__ unsigned parts_magnitude(float x) { return (__float_as_uint(x) << 1) - 1u; }
__device__ __forceinline__ bool parts_tiny(unsigned least) { return least < PARTS_TINY - 1u; }

// The next part of two numbers, which it is taken from: v_cvt_pk_bf16_f32, and two exact subtractions.
__device__ __forceinline__ unsigned take_parts(float& x, float& y) {
    const unsigned b = __builtin_bit_cast(unsigned, __builtin_convertvector(parts_f32x2{x, y}, parts_bf16x2));
    x -= __uint_as_float(b << 16);
    y -= __uint_as_float(b & 0xffff0000u);
    return b;
}

// The parts of eight consecutive numbers: fragments of the 16-bit MFMAs, h in p[0], m in p[1], l in p[2].
__device__ __forceinline__ void split_parts(const parts_f32x4 (&v)[2], parts_u32x4 (&p)[3]) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        float x = v[d >> 1][2 * (d & 1)], y = v[d >> 1][2 * (d & 1) + 1];
#pragma unroll
        for (int i = 0; i < 3; ++i) p[i][d] = take_parts(x, y);
    }
}

}  // namespace sp
