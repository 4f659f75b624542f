// Correctly rounded single-precision quotients and roots in a few fused operations, for
// operands whose range is known (device code only).
#pragma once

#include <hip/hip_runtime.h>

namespace gbr {

// (Each is compared with the general operation by tests/test_gpu_exact.py, the
// first and the last over every float of their ranges.)

// 1 / x, correctly rounded, for 2^-126 <= |x| <= 2^126: the hardware
// reciprocal (1 ulp) and one Newton step in fused arithmetic, three
// instructions instead of the ten of the general division.
__device__ __forceinline__ float rcp_exact(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
}

// a / b, correctly rounded, from r = rcp_exact(b): the quotient's remainder
// corrects it (Markstein 1990).  For b in rcp_exact()'s range, |a| from 2^-100
// to 2^126 and |a / b| from 2^-125 to 2^126, where the quotient is normal and
// the remainder's last bit (2^-47 of a) is a float; or a = 0, whose sign is
// not kept.
__device__ __forceinline__ float div_exact(float a, float b, float r) {
  const float q = a * r;
  return __builtin_fmaf(__builtin_fmaf(-b, q, a), r, q);
}

// sqrt(x), correctly rounded, for 2^-80 <= x <= 2^80
__device__ __forceinline__ float sqrt_exact(float x) {
  const float y = __builtin_amdgcn_rsqf(x), s = x * y;
  return __builtin_fmaf(__builtin_fmaf(-s, s, x), 0.5f * y, s);
}

__device__ __forceinline__ bool in_range(float x, float lo, float hi) {
  return __builtin_amdgcn_fmed3f(fabsf(x), lo, hi) == fabsf(x);
}

}  // namespace gbr
