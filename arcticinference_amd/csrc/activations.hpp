// sigmoid and GELU of the speculator operators on gfx950's transcendental unit.
#pragma once
#include <hip/hip_runtime.h>

namespace arctic {

// sigmoid_f / gelu_erf / gelu_tanh of the reference (sum_lstm.cu:14-26), built on
// the hardware exp2 and reciprocal instructions (1 ulp each) instead of library
// calls: per output element the operator needs three sigmoids and two GELUs, and
// with library expf / erff / IEEE division the arithmetic alone would take longer
// than moving the row through HBM.
__device__ __forceinline__ float fast_exp(float x) {            // e^x
  return __builtin_amdgcn_exp2f(x * 1.4426950408889634f);
}
__device__ __forceinline__ float sigmoid_f(float x) {
  return __builtin_amdgcn_rcpf(1.0f + fast_exp(-x));
}
// gelu(x) = x * Phi(x) = max(x, 0) - |x| q(|x|) with q(z) = Phi(-z) = 2^P(z), P a polynomial of degree 8: one
// transcendental instruction per value.  The rational form of Abramowitz & Stegun 7.1.26 takes two (a reciprocal as
// well) and one more multiply, and where a launch of sum_lstm waits for its arithmetic that shows (us per call in a
// graph, rational form / this one): 7 rows of 4096 4.23 / 4.00, 512 rows of 8192 13.7 / 13.0, 2048 of 2880 21.6 / 20.3.
// P is the best uniform fit of log2 Phi(-z) on [0, 5.8] under the weight max(q max(z, 0.3), 5e-5), as a linear program
// over 6000 points gives it: the error of z q, and in the tail the relative error of q.  Against 64 bits (rational form
// in brackets): 2.6e-8 (5.4e-8) rms over N(0, 1), 2.5e-7 (3.3e-7) at the worst, relative 3e-5 (1.7e-4) where
// |gelu| > 1e-3, 5e-5 (5e-4) at -4 and 2.4e-3 (3.6e-3) at -6.  Beyond 5.8 P goes on falling, from -28.
__device__ __forceinline__ float gelu_erf(float x) {
  const float ax = fabsf(x);
  float p = fmaf(-9.312184374721255e-07f, ax, 1.5563609849778004e-05f);
  p = fmaf(p, ax, -6.800304254284129e-05f);
  p = fmaf(p, ax, -0.0004356678109616041f);
  p = fmaf(p, ax, 0.0074738264083862305f);
  p = fmaf(p, ax, -0.05279786139726639f);
  p = fmaf(p, ax, -0.45910027623176575f);
  p = fmaf(p, ax, -1.1511198282241821f);
  p = fmaf(p, ax, -0.9999997019767761f);
  return fmaf(-ax, __builtin_amdgcn_exp2f(p), fmaxf(x, 0.0f));
}
__device__ __forceinline__ float gelu_tanh(float x) {
  // 0.5 x (1 + tanh(u)) = x * sigmoid(2u),  u = sqrt(2/pi) (x + 0.044715 x^3)
  const float u = 0.79788456080286535588f * fmaf(0.044715f * x * x, x, x);
  return x * sigmoid_f(2.0f * u);
}
template <bool kFastGelu>
__device__ __forceinline__ float gelu(float x) {
  return kFastGelu ? gelu_tanh(x) : gelu_erf(x);
}

}  // namespace arctic
