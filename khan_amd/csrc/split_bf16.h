// A float32 value as the exact sum of three bfloat16 values, for float32 products on the bfloat16 matrix instructions
// (what is formed of them and what it leaves out: dense_first.hip, dense_split_kernel).
#pragma once
#include <hip/hip_runtime.h>

namespace khan {

typedef unsigned u2v __attribute__((ext_vector_type(2)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f2v __attribute__((ext_vector_type(2)));

// two floats -> their three bfloat16 parts, each pair packed into one register (first value in the low half)
__device__ __forceinline__ void split_pair(float x0, float x1, unsigned& p1, unsigned& p2, unsigned& p3)
{
    p1 = __builtin_bit_cast(unsigned, __builtin_convertvector(f2v{x0, x1}, bf16x2));
    const float r0 = x0 - __uint_as_float(p1 << 16), r1 = x1 - __uint_as_float(p1 & 0xffff0000u);
    p2 = __builtin_bit_cast(unsigned, __builtin_convertvector(f2v{r0, r1}, bf16x2));
    const float s0 = r0 - __uint_as_float(p2 << 16), s1 = r1 - __uint_as_float(p2 & 0xffff0000u);
    p3 = __builtin_bit_cast(unsigned, __builtin_convertvector(f2v{s0, s1}, bf16x2));
}

}  // namespace khan
