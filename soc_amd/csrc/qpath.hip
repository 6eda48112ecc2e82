// qpath.hip - rounding of fp32 tensors in device memory to fp16 (weights loaded from device tensors).
#include <algorithm>

#include "kernels.h"

namespace soc {
namespace {

__global__ void k_f32_to_f16(const float* __restrict__ x, size_t n, f16* __restrict__ y) {
  for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
       i += static_cast<size_t>(gridDim.x) * blockDim.x)
    y[i] = static_cast<f16>(x[i]);
}

int blocks_for(size_t n) { return static_cast<int>(std::min<size_t>((n + 255) / 256, 2048)); }

}  // namespace

hipError_t launch_f32_to_f16(const float* x, size_t n, f16* y, hipStream_t s) {
  hipLaunchKernelGGL(k_f32_to_f16, dim3(blocks_for(n)), dim3(256), 0, s, x, n, y);
  return hipGetLastError();
}

}  // namespace soc
