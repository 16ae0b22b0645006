// Reciprocals for the hot loops.  IEEE division compiles to a ~10-instruction
// scale/rcp/Newton/fixup sequence on gfx950; where the divisor is a
// well-scaled positive number (densities, WENO weight sums, cp - R, dx) the
// hardware reciprocal refined by a third-order step (FP64, <= ~1 ulp) or taken
// as is (FP32, 1 ulp) gives the same result to rounding at a third of the
// cost.  Host builds (used to check these headers against the oracle) divide.
#pragma once
#include <math.h>

#include "janc_types.hpp"

namespace jh {

__host__ __device__ __forceinline__ double rcp(double b) {
#if defined(__HIP_DEVICE_COMPILE__)
  // v_rcp_f64 is good to 2^-24.4 (largest error over 2^20 mantissas), so one
  // third-order step r (1 + e + e^2) leaves 2^-73 before its last rounding: an
  // operation less than two Newton steps
  const double r = __builtin_amdgcn_rcp(b);
  const double e = fma(-b, r, 1.0);
  return fma(r, fma(e, e, e), r);
#else
  return 1.0 / b;
#endif
}

__host__ __device__ __forceinline__ float rcp(float b) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rcpf(b);
#else
  return 1.0f / b;
#endif
}

}  // namespace jh
