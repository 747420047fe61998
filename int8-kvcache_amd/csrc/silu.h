// SiLU in fp32, shared by the SwiGLU kernel and the product it is fused into (which must agree bit
// for bit).
#pragma once

#include <hip/hip_runtime.h>

namespace int8kv_loop {

// silu(g) = g / (1 + exp(-g)) without expf's range handling and the IEEE divide (about 35
// instructions an element, in branches whose registers the fused product does not have):
// -g log2(e) as a rounded product plus its rounding error (Cody and Waite's split constant), the
// error applied to exp2 of the product; the hardware's reciprocal refined by one Newton-Raphson
// step and the quotient corrected by its remainder (Markstein).  Over every
// bf16 value with |g| < 87 the result is within 1.35e-7 relative of 64 bits, which is also what
// a correctly rounded exp and divide give.
constexpr float kLog2eHi = 1.44269502162933349609375f;  // log2(e) rounded to fp32, and the rest
constexpr float kLog2eLo = 1.925963033500011e-08f;
constexpr float kLn2 = 0.693147180559945f;
constexpr float kSiluMiddle = 87.0f;

__device__ __forceinline__ float silu_middle(float g) {
  const float t = -g * kLog2eHi;
  const float lo = fmaf(-g, kLog2eHi, -t) - g * kLog2eLo;
  const float x = __builtin_amdgcn_exp2f(t);
  const float d = 1.0f + fmaf(x * kLn2, lo, x);
  float r = __builtin_amdgcn_rcpf(d);
  r = fmaf(fmaf(-d, r, 1.0f), r, r);
  const float q = g * r;
  return fmaf(fmaf(-d, q, g), r, q);
}

// The rest: g itself above (1 + exp(-g) is 1 there), g exp(g) below, with exp(g) 2^64 in range
// (1 + exp(-g) is exp(-g) there), and -0 from where exp(-g) overflows fp32, as g / infinity.  -inf
// gives NaN there too (-inf / inf, as torch's silu), and a NaN stays one.
__device__ __forceinline__ float silu_ends(float g) {
  const float t = g * kLog2eHi;
  const float lo = fmaf(g, kLog2eHi, -t) + g * kLog2eLo;
  const float x = __builtin_amdgcn_exp2f(t + 64.0f);
  const float low = g * fmaf(x * kLn2, lo, x) * 0x1p-64f;
  return g > 0.0f ? g : (g < -88.7228394f ? g * 0.0f : low);
}

__device__ __forceinline__ float silu(float g) {
  return fabsf(g) < kSiluMiddle ? silu_middle(g) : silu_ends(g);
}

// y[i] = silu(g[i]), one branch for the rare elements outside the middle.
template <int N>
__device__ __forceinline__ void silu(const float (&g)[N], float (&y)[N]) {
  bool all = true;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    y[i] = silu_middle(g[i]);
    all &= fabsf(g[i]) < kSiluMiddle;
  }
  if (!all) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (!(fabsf(g[i]) < kSiluMiddle)) y[i] = silu_ends(g[i]);
  }
}

}  // namespace int8kv_loop
