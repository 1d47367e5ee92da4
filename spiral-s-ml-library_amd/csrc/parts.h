// A f32 as the sum of three bf16 numbers, for products on the bf16 matrix pipe.
//
// Every f32 is the exact sum of three bf16 numbers, x = h + m + l: h is x rounded to bf16, m what is left rounded to bf16, l
// the rest (8 significant bits each and two signs: 24 bits and more).  A product of two f32 is then nine products of bf16, of
// which the smallest, l l, is below 2^-33 of it and left out.
//   How the eight are added up decides what the sum is worth.  Where the bf16 MFMAs add to an accumulator that is not zero they cut
// off what lies below the last bit of the larger (towards minus infinity; up to 2 ulp, f32 MFMAs round to nearest).  So the products
// h h of one MFMA, 16 or 32 of K, are added up from zero, and to those of the other MFMAs by the vector ALU, which rounds to
// nearest; the other seven, 2^-8 of the whole, have an accumulator of their own that is added at the end.  A single product is
// rounded once, as the f32 pipe does it (but for one in a thousand, where what is lost in the small sum tips it), and sums have fewer
// roundings than there.  Layer 1 of the ensemble kernel, K = 128, error against float64 (2-norm: f32 MFMAs / so / six products in
// one accumulator): N(0, 1) inputs 2.03e-7 / 5.9e-8 / 1.62e-7, relu of them 1.39e-7 / 4.9e-8 / 1.51e-7, a fifth ones and else zeros
// 9.3e-8 / 2.5e-8 / 7.8e-8, eight non-zero numbers a row 5.3e-8 / 2.8e-8 / 9.5e-8, two 3.1e-8 / 2.5e-8 / 5.0e-8, one 2.53e-8 / 2.53e-8 / 3.45e-8.
#pragma once
#include "common.h"

namespace sp {

typedef __bf16 parts_bf16x2 __attribute__((ext_vector_type(2)));
typedef float parts_f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned parts_u32x4 __attribute__((ext_vector_type(4)));
typedef float parts_f32x4 __attribute__((ext_vector_type(4)));

// Products of parts, weights x inputs, in the order in which they are added up: the second to the last to the small sum.
constexpr int PARTS_W[8] = {0, 2, 1, 2, 0, 1, 1, 0}, PARTS_X[8] = {0, 1, 2, 0, 2, 1, 0, 1};

// l holds the last bit of a number as long as that is no smaller than the smallest bf16, 2^-133 (the pipe keeps subnormal numbers):
// inputs are taken times 2^16, where every f32 is in range, and weights times 2^-16, where all from 2^-94 up are.  If there are
// smaller ones, the weights are taken times 2^16, too, and the sums times 2^-32.  Rows of inputs above 2^60, and weights above
// that (with small ones among them, above 2^28), whose sums might overflow in parts, go through f32 MFMAs.
constexpr float PARTS_X_SCALE = 0x1p16f, PARTS_W_SCALE = 0x1p-16f, PARTS_W_SCALE_SMALL = 0x1p16f, PARTS_UNSCALE_SMALL = 0x1p-32f, PARTS_MOST = 0x1p60f;
// The smallest non-zero 2 |w|, in bits and less one (zeros wrap to the largest).
constexpr unsigned PARTS_TINY = (127u - 94u) << 24;
__device__ __forceinline__ unsigned parts_magnitude(float w) { return (__float_as_uint(w) << 1) - 1u; }

struct PartsWeights {                     // what the weights seen ask for (NaN: a NaN either way)
    unsigned least = 0xffffffffu;
    float most = 0.f;
    __device__ __forceinline__ void take(float w) {
        const unsigned m = parts_magnitude(w);
        least = m < least ? m : least;
        most = fmaxf(most, fabsf(w));
    }
    __device__ __forceinline__ bool small() const { return least < PARTS_TINY - 1u; }
    __device__ __forceinline__ bool large() const { return most > 0x1p28f; }
    __device__ __forceinline__ bool wide() const { return most > PARTS_MOST; }
};

// max(most, |x|, |y|), a NaN passed over.
__device__ __forceinline__ float parts_most(float most, float x, float y) {
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(most) : "v"(x), "v"(y));
    return most;
}

// The next part of two numbers, which it is taken from: v_cvt_pk_bf16_f32, and two exact subtractions.
__device__ __forceinline__ unsigned take_parts(float& x, float& y) {
    const unsigned b = __builtin_bit_cast(unsigned, __builtin_convertvector(parts_f32x2{x, y}, parts_bf16x2));
    x -= __uint_as_float(b << 16);
    y -= __uint_as_float(b & 0xffff0000u);
    return b;
}

// The parts of scale times eight consecutive numbers: fragments of the 16-bit MFMAs, h in p[0], m in p[1], l in p[2].
__device__ __forceinline__ void split_parts(const parts_f32x4 (&v)[2], float scale, parts_u32x4 (&p)[3]) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        float x = v[d >> 1][2 * (d & 1)] * scale, y = v[d >> 1][2 * (d & 1) + 1] * scale;
#pragma unroll
        for (int i = 0; i < 3; ++i) p[i][d] = take_parts(x, y);
    }
}

}  // namespace sp
