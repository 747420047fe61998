// SiLU in fp32, shared by the SwiGLU kernel and the product it is fused into (which must agree bit
// for bit).
#pragma once

#include <hip/hip_runtime.h>

namespace int8kv_loop {

// silu(g) = g / (1 + exp(-g)) for |g| < kSiluFast without the range checks of expf and the IEEE
// divide (about 35 instructions an element with them): -g log2(e) as a rounded product plus its
// rounding error, the error applied to exp2 of the product; the reciprocal refined once and the
// quotient corrected by its remainder.  Over every bf16 value of that range the result is within
// 1.35e-7 relative of 64 bits, which is also what a correctly rounded exp and divide give.
constexpr float kSiluFast = 80.0f;

__device__ __forceinline__ float silu_fast(float g) {
  const float kL = 1.44269502162933349609375f;  // log2(e) rounded to fp32, and the rest
  const float kLlo = 1.925963033500011e-08f;
  const float t = -g * kL;
  const float lo = fmaf(-g, kL, -t) - g * kLlo;
  const float x = __builtin_amdgcn_exp2f(t);
  const float d = 1.0f + fmaf(x * 0.693147180559945f, lo, x);
  float r = __builtin_amdgcn_rcpf(d);
  r = fmaf(fmaf(-d, r, 1.0f), r, r);
  const float q = g * r;
  return fmaf(fmaf(-d, q, g), r, q);
}

// y[i] = silu(g[i]); the elements outside the fast range (and NaN) take expf and the divide.
template <int N>
__device__ __forceinline__ void silu(const float (&g)[N], float (&y)[N]) {
  bool all = true;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    y[i] = silu_fast(g[i]);
    all &= fabsf(g[i]) < kSiluFast;
  }
  if (!all) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (!(fabsf(g[i]) < kSiluFast)) y[i] = g[i] / (1.0f + expf(-g[i]));
  }
}

}  // namespace int8kv_loop
