// A float32 value as the sum of two half-precision values, x = h + 2^-11 l, for float32 products on the half-precision matrix
// instructions: three of them form h h' + 2^-11 (h l' + l h') (what that leaves out: dense_fused.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace khan {

typedef unsigned u2v __attribute__((ext_vector_type(2)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f2v __attribute__((ext_vector_type(2)));

constexpr float kResidualScale = 2048.0f, kResidualBack = 1.0f / 2048.0f;      // 2^11

// two floats -> their two half-precision parts (the value rounded, and 2^11 times what the rounding left), each pair
// packed into one register (first value in the low half).  Both differences are exact in float32.
__device__ __forceinline__ void split_pair(float x0, float x1, unsigned& p1, unsigned& p2)
{
    const h2v h = __builtin_convertvector(f2v{x0, x1}, h2v);
    p1 = __builtin_bit_cast(unsigned, h);
    // 2^11 x - 2^11 h in one fused multiply-add that reads h and writes half precision as they are (both products are exact,
    // and so is the difference)
    h2v l;
    l[0] = static_cast<_Float16>(fmaf(static_cast<float>(h[0]), -kResidualScale, x0 * kResidualScale));
    l[1] = static_cast<_Float16>(fmaf(static_cast<float>(h[1]), -kResidualScale, x1 * kResidualScale));
    p2 = __builtin_bit_cast(unsigned, l);
}

}  // namespace khan
