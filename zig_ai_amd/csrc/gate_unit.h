// The gated units that products apply to their own 32-bit sums: act(v) * u of a gate and an up column.
#pragma once

#include "common.h"

// 1 / (1 + exp(-x)).  EXACT: to the last bit of 32-bit division and expf.  Otherwise in the hardware's
// exponential and reciprocal, some 12 clocks an element and lane instead of 31 (a wave of the wide products has
// 128 of them to do while the matrix cores stand still): within 1e-6 of it for |x| up to 20, a four-thousandth
// of what rounding the unit to bfloat16 leaves; infinities and NaN as the other.
template <bool EXACT>
__device__ __forceinline__ float unit_sigmoid(float x) {
  if constexpr (EXACT) return 1.0f / (1.0f + expf(-x));
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x));
}

// KIND 1: silu, 2: the tanh form of gelu, 3: v * sigmoid(slope * v) * (u + offset) with v and u bounded
// (bound > 0).  For results in bfloat16 EXACT is left out.
template <int KIND, bool EXACT>
__device__ __forceinline__ float gated_value(float v, float u, float bound, float slope, float offset) {
  if constexpr (KIND == 3) {
    v = bound > 0.f ? fminf(v, bound) : v;
    u = bound > 0.f ? fminf(fmaxf(u, -bound), bound) : u;
    return v * unit_sigmoid<EXACT>(slope * v) * (u + offset);
  }
  if constexpr (KIND == 2)
    return 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v))) * u;
  return v * unit_sigmoid<EXACT>(v) * u;
}
