// Entry points through which tests look at the arithmetic of device functions.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/gatehip.h"
#include "gh_device.h"

namespace {

__global__ void __launch_bounds__(256) quotient_kernel(const float *__restrict__ a, const float *__restrict__ b,
                                                       int64_t n, float *__restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    out[i] = gh::quotient(a[i], b[i]);
}

}  // namespace

extern "C" int gh_quotient(const float *a, const float *b, int64_t n, float *out, void *stream) {
  if (!a || !b || !out || n < 0) return GH_EINVAL;
  if (n == 0) return GH_OK;
  const unsigned grid = (unsigned)std::min<int64_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(quotient_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream, a, b, n, out);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}
