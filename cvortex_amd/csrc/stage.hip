// stage.hip -- copies between pinned host memory and the device by a kernel.
//
// A small call on host arrays is bound by latencies: for a small pinned copy HIP
// launches a kernel of its own, with barriers and a completion signal around it,
// which takes three to six microseconds more than this one, and above about 50 KB
// it sets up a DMA engine.  Copy -> this kernel in, and out too or (up to 64 KB)
// the outputs written straight to host memory, us a call: 3D velocity of 1000
// particles 31.5 -> 25.0, of 5000 60.8 -> 49.7, exchange of 1000 on 2000 40.3 ->
// 28.1, 1000 filaments on 3000 targets 47.9 -> 33.9, vorticity of 6000 on 9000
// 106 -> 83, 2D velocity of 8000 62.6 -> 51.5; at 0.65 MB in 147 -> 140, at 1 MB
// (30000 2D particles) 290 -> 285, where the lines of kStageMax stand.
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace cvtx {

namespace {

__global__ __launch_bounds__(256) void stage_kernel(const float4* __restrict__ src,
                                                    float4* __restrict__ dst, int n, int tail) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = src[i];
  if (i < tail) ((float*)(dst + n))[i] = ((const float*)(src + n))[i];
}

}  // namespace

hipError_t launch_stage(void* dst, const void* src, size_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  if (bytes % 4 != 0 || bytes > kStageMax) return hipErrorInvalidValue;
  const int n = (int)(bytes / 16), tail = (int)(bytes % 16 / 4);
  hipLaunchKernelGGL(stage_kernel, dim3(n / 256 + 1), dim3(256), 0, s, (const float4*)src,
                     (float4*)dst, n, tail);
  return hipGetLastError();
}

}  // namespace cvtx
