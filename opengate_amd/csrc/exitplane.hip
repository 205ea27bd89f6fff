// Learned exit-plane source: generator noise and the decoder from generator outputs
// to phase-space records.
//
// gh_gaussian_bf16: N(0,1) noise for the generator input, one Philox4x32-10 block
// (key = seed, counter = (row lo, row hi, "NOIS", column/4)) per 4 columns of a row,
// Box-Muller on the two uniform pairs. A row depends only on (seed, row index), so
// chunked generation reproduces one big batch.
//
// gh_exitplane_decode: the generator emits 6 values per photon in a Gaussianised
// space: (E, x, y, u', v', w'). Each value is mapped back through its feature's
// quantile table (knots at equally spaced Gaussian values g_k in [-g_max, g_max],
// linear between knots, clamped at the ends), then
//   position  (x, y, plane_z) on the exit plane,
//   direction d = u' e1 + v' e2 + w' n (normalised), with n the unit vector from the
//             focal point to (x, y, plane_z) and (e1, e2, n) the right-handed frame
//             e1 = (nx nz, ny nz, -up)/up, e2 = (-ny, nx, 0)/up, up = |(nx, ny)|
//             (up -> 0: e1 = (nz, 0, 0), e2 = (0, 1, 0)).
// Photons that travel along the ray from the focal point therefore have
// (u', v', w') = (0, 0, 1): the generator learns deviations from the point-source
// geometry instead of the steep position-direction correlation itself.
// Records are written as 8 float arrays (x, y, z, u, v, w, E, weight) shifted by an
// offset into the frame of the next simulation.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/gatehip.h"
#include "exitplane.h"

namespace {

__global__ void __launch_bounds__(256) gaussian_bf16_kernel(uint32_t k0, uint32_t k1, uint64_t first, int64_t n,
                                                            int cols, int ld, __bf16 *__restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += stride) {
    for (int c0 = 0; c0 < ld; c0 += 4) {
      float g[4];
      ep::noise4(first + (uint64_t)r, (uint32_t)(c0 >> 2), k0, k1, g);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int c = c0 + j;
        if (c < ld) out[r * ld + c] = (__bf16)(c < cols ? g[j] : 0.0f);
      }
    }
  }
}

__global__ void __launch_bounds__(256) exitplane_decode_kernel(const float *__restrict__ Z, int64_t ldz, int64_t n,
                                                               ep::Decode d) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    float z[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) z[k] = Z[i * ldz + k];
    ep::decode(d, i, z);
  }
}

int grid_for(int64_t n) {
  int dev = 0, n_cu = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
  const int64_t want = (n + 255) / 256;
  return (int)std::max<int64_t>(1, std::min<int64_t>(want, (int64_t)n_cu * 16));
}

}  // namespace

extern "C" int gh_gaussian_bf16(uint64_t seed, uint64_t first_row, int64_t n_rows, int32_t n_cols, int32_t ld,
                                void *out, void *stream) {
  if (!out || n_rows < 0 || n_cols < 0 || ld < n_cols || ld <= 0) return GH_EINVAL;
  if (n_rows == 0) return GH_OK;
  hipLaunchKernelGGL(gaussian_bf16_kernel, dim3(grid_for(n_rows)), dim3(256), 0, (hipStream_t)stream, (uint32_t)seed,
                     (uint32_t)(seed >> 32), first_row, n_rows, (int)n_cols, (int)ld, (__bf16 *)out);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}

extern "C" int gh_exitplane_decode(const float *Z, int64_t ldz, int64_t n, const float *qtab, int32_t n_knots,
                                   float g_max, const float focal[3], float plane_z, const float offset[3],
                                   float weight, float *const out[8], void *stream) {
  if (!Z || !qtab || !focal || !offset || !out || n < 0 || ldz < 6 || n_knots < 2 || !(g_max > 0.0f))
    return GH_EINVAL;
  for (int k = 0; k < 8; ++k)
    if (!out[k]) return GH_EINVAL;
  if (n == 0) return GH_OK;
  ep::Decode d{qtab, (int)n_knots, (float)(n_knots - 1) / (2.0f * g_max), g_max,
               {focal[0], focal[1], focal[2], plane_z, offset[0], offset[1], offset[2], weight}, {}};
  for (int k = 0; k < 8; ++k) d.out[k] = out[k];
  hipLaunchKernelGGL(exitplane_decode_kernel, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, Z, ldz, n, d);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}
