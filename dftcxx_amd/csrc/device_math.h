// Reciprocals in FP64 from the hardware estimates.
#ifndef DFTGRID_DEVICE_MATH_H
#define DFTGRID_DEVICE_MATH_H

#include <hip/hip_runtime.h>

namespace dg {

// 1/sqrt(x) and 1/x from the hardware estimates (about 2^-26) and two Newton steps.
__device__ __forceinline__ double rsqrt64(double x) {
  double y = __builtin_amdgcn_rsq(x);
  for (int k = 0; k < 2; ++k) y = y * __fma_rn(-0.5 * x * y, y, 1.5);
  return y;
}
__device__ __forceinline__ double rcp64(double x) {
  double y = __builtin_amdgcn_rcp(x);
  for (int k = 0; k < 2; ++k) y = __fma_rn(y, __fma_rn(-x, y, 1.0), y);
  return y;
}

}  // namespace dg

#endif
