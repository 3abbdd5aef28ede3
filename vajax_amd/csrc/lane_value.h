// One lane's value for a whole wavefront, shared by the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace vjx {

// Lane `lane`'s value of v (lane uniform across the wavefront).
__device__ __forceinline__ double lane_value(double v, int lane) {
  const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
  const unsigned int lo = (unsigned int)__builtin_amdgcn_readlane((int)(unsigned int)bits, lane);
  const unsigned int hi =
      (unsigned int)__builtin_amdgcn_readlane((int)(unsigned int)(bits >> 32), lane);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

}  // namespace vjx
