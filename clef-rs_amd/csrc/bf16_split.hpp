// Exact split of f32 values into three bf16 values (f32 products on the bf16
// matrix cores: gemm_f32.hpp, attention_f32.hpp).
#pragma once
#include "common.hpp"

namespace clef {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));

// x = hi + mid + lo exactly, each a bf16: round to nearest takes 8 bits, and
// what is left of a 24-bit significand after two of them fits a third.
__device__ __forceinline__ void split8(const float4_t& a, const float4_t& b, bf16x8& hi, bf16x8& mid, bf16x8& lo) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float2_t x = e < 2 ? float2_t{a[2 * e], a[2 * e + 1]} : float2_t{b[2 * e - 4], b[2 * e - 3]};
    const bf16x2 h = __builtin_convertvector(x, bf16x2);
    const float2_t r = x - __builtin_convertvector(h, float2_t);
    const bf16x2 m = __builtin_convertvector(r, bf16x2);
    const bf16x2 l = __builtin_convertvector(r - __builtin_convertvector(m, float2_t), bf16x2);
    hi[2 * e] = h[0], hi[2 * e + 1] = h[1];
    mid[2 * e] = m[0], mid[2 * e + 1] = m[1];
    lo[2 * e] = l[0], lo[2 * e + 1] = l[1];
  }
}

}  // namespace clef
