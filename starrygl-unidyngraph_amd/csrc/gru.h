// GRU gate combination shared by the memory-update kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace sgl {

// PyTorch order r, z, n:
//   r = s(gi_r + gh_r), z = s(gi_z + gh_z), n = tanh(gi_n + r * gh_n),
//   h' = (1 - z) * n + z * h
__device__ __forceinline__ float gru_combine(float gir, float giz, float gin, float ghr, float ghz,
                                             float ghn, float h) {
  const float r = 1.f / (1.f + expf(-(gir + ghr)));
  const float z = 1.f / (1.f + expf(-(giz + ghz)));
  const float n = tanhf(gin + r * ghn);
  return (1.f - z) * n + z * h;
}

}  // namespace sgl
