// GELU of the GEGLU kernels (geglu.hip and the fused projection in geglu_linear.hip), so
// both compute bitwise the same gelu(a) and gelu'(a).
//   tanh form (the reference's _gelu_parts, library/geglu.py:20-24):
//     z = sqrt(2/pi) (a + 0.044715 a^3);  gelu = 0.5 a (1 + tanh z) = a s,  s = 1 / (1 + e^{-2z})
//   erf form (torch.nn.functional.gelu(approximate="none")):
//     gelu = 0.5 a (1 + erf(a / sqrt 2)),  gelu' = 0.5 (1 + erf(a / sqrt 2)) + a exp(-a^2 / 2) / sqrt(2 pi)
#pragma once

#include <hip/hip_runtime.h>

#include "krsi_device.h"

namespace krsi {
namespace gelu_detail {

constexpr float kTwoSqrt2OverPi = 1.5957691216057308f;    // 2 sqrt(2/pi)
constexpr float kTwoSqrt2OverPiK3 = 0.21406444881780073f;  // 2 sqrt(2/pi) * 3 * 0.044715
constexpr float kNegTwoZ = -2.3022081983814324f;           // -2 sqrt(2/pi) log2 e
constexpr float kNegTwoZK = -0.10294323959062575f;         // -2 sqrt(2/pi) log2 e * 0.044715
constexpr float kInvSqrt2 = 0.70710678118654752f;
constexpr float kInvSqrt2Pi = 0.3989422804014327f;
constexpr float kLog2eG = 1.4426950408889634f;

// The logistic form of (1 + tanh z) / 2, z = sqrt(2/pi) (a + 0.044715 a^3): one exp and one
// reciprocal in place of the division of 1 - 2 / (e^{2z} + 1), and no cancellation for a < 0
// (e^{-2z} overflows to +inf there and s is exactly 0). The hardware reciprocal is off by one fp32
// ulp, far below half a 16-bit ulp of gelu; fp32 divides.
template <int DT>
__device__ __forceinline__ float tanh_gate(float a) {
  const float d = 1.0f + __builtin_amdgcn_exp2f(a * __builtin_fmaf(a * a, kNegTwoZK, kNegTwoZ));
  if constexpr (DT == kF32) return 1.0f / d;
  return __builtin_amdgcn_rcpf(d);
}

// erf by Abramowitz & Stegun, Handbook of Mathematical Functions, 7.1.26:
// erf(x) = 1 - t (a1 + t (a2 + t (a3 + t (a4 + t a5)))) e^{-x^2}, t = 1 / (1 + p x), x >= 0,
// absolute error <= 1.5e-7 (<= 6e-7 evaluated in fp32), far below a bf16 ulp of the output.
// Returns erf(a / sqrt 2); ex must be e^{-a^2 / 2}, which gelu' needs as well.
__device__ __forceinline__ float erf_as(float a, float ex) {
  const float x = fabsf(a) * kInvSqrt2;
  const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3275911f, x, 1.0f));
  float q = __builtin_fmaf(1.061405429f, t, -1.453152027f);
  q = __builtin_fmaf(q, t, 1.421413741f);
  q = __builtin_fmaf(q, t, -0.284496736f);
  q = __builtin_fmaf(q, t, 0.254829592f);
  return copysignf(1.0f - q * t * ex, a);
}
__device__ __forceinline__ float exp_half_sq(float a) {
  return __builtin_amdgcn_exp2f(-0.5f * kLog2eG * a * a);
}

template <int DT, bool TANH>
__device__ __forceinline__ float gelu_fwd(float a) {
  if (TANH) return a * tanh_gate<DT>(a);
  return 0.5f * a * (1.0f + erf_as(a, exp_half_sq(a)));
}

// Returns gelu(a) and writes gelu'(a) to d.
template <int DT, bool TANH>
__device__ __forceinline__ float gelu_fwd_bwd(float a, float& d) {
  if (TANH) {
    // s' = s (1 - s) 2 z', z' = sqrt(2/pi) (1 + 3 * 0.044715 a^2).
    const float s = tanh_gate<DT>(a);
    const float gel = a * s;
    d = __builtin_fmaf(gel * (1.0f - s), __builtin_fmaf(a * a, kTwoSqrt2OverPiK3, kTwoSqrt2OverPi), s);
    return gel;
  }
  const float ex = exp_half_sq(a);
  const float e = erf_as(a, ex);
  const float pdf = ex * kInvSqrt2Pi;
  d = 0.5f * (1.0f + e) + a * pdf;
  return 0.5f * a * (1.0f + e);  // the forward's expression, so bf16(gelu) matches it
}

}  // namespace gelu_detail

using gelu_detail::gelu_fwd;
using gelu_detail::gelu_fwd_bwd;

}  // namespace krsi
