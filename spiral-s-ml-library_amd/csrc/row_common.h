// Arithmetic the row primitives and the fused stacks with a row head share, operation for operation.
#pragma once
#include "common.h"

#pragma clang fp contract(off)

namespace sp {

// exp(x) = 2^(x * log2 e) on the hardware exp2 unit; relative error about 1e-6 for |x| < 20.
__device__ __forceinline__ float fast_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896340736f); }

__device__ __forceinline__ float sum4(const float (&v)[4]) { return ((v[0] + v[1]) + v[2]) + v[3]; }

// x / s for many x and one s as x * scale * (1 / (s * scale)): one division per row, and `scale` (a power of two, so
// both products by it are exact) keeps the reciprocal finite when s lies below 2^-126, where 1 / s alone would be
// +inf and every quotient inf or NaN.  The quotients differ from a correctly rounded x / s by at most one unit in
// the last place.
struct RowDivisor {
    float scale, inv;
    __device__ __forceinline__ explicit RowDivisor(float s) {
        scale = fabsf(s) < 4.7019774e-38f ? 1.8446744e19f : 1.f;     // below 2^-124: times 2^64
        inv = 1.f / (s * scale);
    }
    __device__ __forceinline__ float operator()(float x) const { return (x * scale) * inv; }
};

}  // namespace sp
