// CELU of the float32 layers (net_layers.hip, net_chain.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace khan {

// exp(x) - 1 for x <= 0 to 1.5 units in the last place (exp(x) - 1 as written is 0 from -3e-8 up, where a layer's output then
// counts as its positive side, and 0.6 % off at -1e-5): x = k ln 2 + f with |f| <= ln 2 / 2 (k from the bits of x log2 e +
// 1.5 2^23, ln 2 in two parts), exp(f) - 1 = f + f^2 r(f) with r interpolated at Chebyshev points, and 2^k (exp(f) - 1) +
// (2^k - 1).  Below -88 it is -1, in float32 too; x is not NaN.  Twelve vector instructions more than the other form per
// activation, 9 % of a layer's time (47,000 rows 256 -> 256: 39.7 -> 43.2 us).
__device__ __forceinline__ float expm1_down(float x)
{
    x = fmaxf(x, -88.0f);
    const float shifted = fmaf(x, 0x1.715476p+0f, 12582912.0f), k = shifted - 12582912.0f;
    const float two_k = __int_as_float((__float_as_int(shifted) << 23) + 0x3f800000);
    const float f = fmaf(k, 0x1.05c610p-29f, fmaf(k, -0x1.62e430p-1f, x));
    float r = fmaf(0x1.6b4822p-10f, f, 0x1.12294ep-7f);
    r = fmaf(r, f, 0x1.55574ap-5f);
    r = fmaf(r, f, 0x1.5554aep-3f);
    r = fmaf(r, f, 0x1.fffffep-2f);
    return fmaf(two_k, fmaf(r * f, f, f), two_k - 1.0f);
}

// celu(z) = z for z >= 0, alpha (exp(z / alpha) - 1) below (inv = 1 / alpha); _absolute: with an absolute error of 2^-24 alpha
__device__ __forceinline__ float celu_exact(float z, float alpha, float inv) { return z < 0.f ? alpha * expm1_down(z * inv) : z; }
__device__ __forceinline__ float celu_absolute(float z, float alpha, float inv) { return z >= 0.f ? z : alpha * (__expf(z * inv) - 1.0f); }

}  // namespace khan
