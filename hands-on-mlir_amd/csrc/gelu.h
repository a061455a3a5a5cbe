// The two forms of GELU as every GEMM epilogue computes them.
#pragma once

#include <hip/hip_runtime.h>

namespace hom {

// GELU(x) = 0.5 x (1 + erf(x / sqrt 2)) = max(x, 0) - 0.5 |x| erfc(|x| / sqrt 2)
// (x >= 0: 1 + erf = 2 - erfc; x < 0: 1 + erf = erfc(|z|); no cancellation on
// the negative side), with erfc(a / sqrt 2) = 2^P(a): P is the degree-6 least
// squares fit of log2 erfc(a / sqrt 2) on [0, 8], weighted by the sensitivity
// of GELU to it.  Absolute error <= 2.7e-7 over fp32 inputs (the fp32 rounding
// of the result itself near |x| = 4), at most one fp16 ulp away from the
// exactly rounded value.  Beyond a = 8 the factor stays at 2^P(8) ~ 1e-15.
// Six FMAs and one exp2: the epilogue runs when no MFMA work is left to hide
// it, so its instruction count is wall time; the library erff costs 3x this.
__device__ __forceinline__ float geluErf(float x) {
  const float ax = fabsf(x);
  const float a = fminf(ax, 8.0f);
  float P = fmaf(3.448796997e-05f, a, -7.812886615e-04f);
  P = fmaf(P, a, 8.119936101e-03f);
  P = fmaf(P, a, -5.347220227e-02f);
  P = fmaf(P, a, -4.587264359e-01f);
  P = fmaf(P, a, -1.151216269e+00f);
  P = fmaf(P, a, 8.451195754e-06f);
  return fmaf(-0.5f * ax, __builtin_amdgcn_exp2f(P), fmaxf(x, 0.0f));
}
// 0.5 x (1 + tanh(u)) == x / (1 + exp(-2u)), u = sqrt(2/pi) (x + 0.044715 x^3)
__device__ __forceinline__ float geluTanh(float x) {
  // exp(-2u) = exp2(-2 log2(e) u) = exp2(x (c1 + c3 x^2)) with the constants
  // folded: c1 = -2 log2(e) sqrt(2/pi), c3 = 0.044715 c1 (three multiplies
  // fewer per output; the epilogue's instruction count is wall time).
  // Large negative x gives x * rcp(inf) = -0.
  const float w = fmaf(x * x, -0.1029432397f, -2.3022081983f);
  const float e = __builtin_amdgcn_exp2f(x * w);
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}

} // namespace hom
