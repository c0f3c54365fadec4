// The gated units that products apply to their own 32-bit sums: act(v) * u of a gate and an up column.
#pragma once

#include "common.h"

// 1 / (1 + exp(-x)).  EXACT: 32-bit division and expf as they are.  Otherwise the same value without what those do
// for arguments that do not come here (a wave of the wide products has 128 of them a lane to do while the matrix cores
// stand still): exp(y) as 2^n 2^f, y log2(e) = n + f in two parts, and one step of Newton's on the reciprocal.  All
// is 2^-36 times itself until the end, so that nothing overflows and a result below the normal range has a
// normal one to be rounded from.  Over all 2^32 values of x it has the other's bits but for 13 that differ by one
// unit, and those below -87.3 (less than 1.2e-38), where it goes on to the smallest number and the other stops
// at 2^-128.  A NaN gives 0, which is NaN again times the v it comes from.
template <bool EXACT>
__device__ __forceinline__ float unit_sigmoid(float x) {
#pragma clang fp contract(off)
  if constexpr (EXACT) return 1.0f / (1.0f + expf(-x));
  constexpr float WHOLE = 12582912.0f - 36.0f;      // 1.5 x 2^23: its sum with p ends in the bits of n - 36
  const float y = -__builtin_amdgcn_fmed3f(x, -110.f, 60.f), p = y * 1.44269502f, up = p + WHOLE, n = up - WHOLE;
  const float low = __builtin_fmaf(y, 1.92596299e-8f, __builtin_fmaf(y, 1.44269502f, -p));
  const float t = __builtin_amdgcn_exp2f((p - n) + low);
  const float e = __uint_as_float(__float_as_uint(t) + (__float_as_uint(up) << 23));
  const float d = e + 0x1p-36f, r = __builtin_amdgcn_rcpf(d);
  return __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r) * 0x1p-36f;
}

// KIND 1: silu, 2: the tanh form of gelu, 3: v * sigmoid(slope * v) * (u + offset) with v and u bounded
// (bound > 0).  For results in bfloat16 EXACT is left out.  (us, with EXACT and without: gated products of the wide
// tiles 2 x 8192 x 2048 at 2,048 rows 114 and 109, 2 x 4608 x 1024 at 1,037 rows 31 and 28; the unit by itself on 8,192
// outputs of 1,037 rows 11.0 and 9.9.  The hardware's exponential of a rounded product and its reciprocal as they are,
// 106, 26 and 9.1, were off by up to 1e-6 at |x| of 20 and 4e-6 at 87.)
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
