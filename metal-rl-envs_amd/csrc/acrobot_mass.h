// The entries of Acrobot's mass matrix that depend on c2 = cos(theta2) alone, and their quotients
// (acrobot_np.py:64-84; each constant's defining expression is beside it).
#pragma once

#include "hipenvs_device.h"

namespace hipenvs {
namespace ac {

constexpr float D1_C0 = 0x1p-2f;              // float32(1.0 * 0.5**2)
constexpr float D1_C1 = 0x1.4p+0f;            // float32(1.0**2 + 0.5**2)
constexpr float D2_C0 = 0x1p-2f;              // float32(0.5**2)
constexpr float D2_C1 = 0x1p-1f;              // float32(1.0 * 0.5)

__device__ __forceinline__ float mass_d1(float c2) { return ((D1_C0 + (D1_C1 + c2)) + 1.0f) + 1.0f; }
__device__ __forceinline__ float mass_d2(float c2) { return (D2_C0 + D2_C1 * c2) + 1.0f; }

// a / d1 for a = d2 or d2 * d2, with r the hardware's reciprocal estimate of d1: the estimate's
// quotient and one residual correction. Both quotients are functions of c2 alone: equal to the
// IEEE division for every float32 c2 in [-kMassRange, kMassRange], where d1 lies in [2.5, 4.5]
// and d2 in [0.75, 1.75] (hipenvs_arith_check, run by the GPU tests), and NaN with it for a NaN.
// det_sincos's cosine is in [-1, 1] for angles up to about 2^50; past them it can be of any size,
// d1 0 or infinite, and the quotient is IEEE division's only with kInRange false. Four
// instructions with the estimate where the IEEE division takes eleven, one after the other, on
// the chain of each of the four derivatives of a step: rollout (16 lanes a member, P = 4,096,
// H = 32, 500 steps) 879 -> 826 us; the step at N = 2^20 takes 19.1 us, as it did through d1's
// float64 reciprocal (19.2), and 22.5 with IEEE division.
constexpr float kMassRange = 1.5f;

template <bool kInRange = true>
__device__ __forceinline__ float mass_quotient(float a, float d1, float r) {
  if constexpr (!kInRange) return a / d1;
  const float q = a * r;
  return __builtin_fmaf(__builtin_fmaf(-d1, q, a), r, q);
}

}  // namespace ac
}  // namespace hipenvs
