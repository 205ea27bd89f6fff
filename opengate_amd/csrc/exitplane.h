// Device code of the learned exit-plane source that its own kernels (exitplane.hip) and the
// generator's fused forms (mlp.hip) share: noise and decoder.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#include "gh_device.h"

namespace ep {

constexpr uint32_t NOISE_TAG = 0x4E4F4953u;  // "NOIS"

// columns 4 block .. 4 block + 3 of noise row `row`: one Philox4x32-10 block, Box-Muller on
// the two uniform pairs
__device__ __forceinline__ void noise4(uint64_t row, uint32_t block, uint32_t k0, uint32_t k1, float (&g)[4]) {
  uint32_t x0 = (uint32_t)row, x1 = (uint32_t)(row >> 32), x2 = NOISE_TAG, x3 = block;
  gh::philox10(x0, x1, x2, x3, k0, k1);
  const float u0 = (float)((x0 >> 8) | 1u) * 0x1p-24f, u1 = (float)((x1 >> 8) | 1u) * 0x1p-24f;
  const float u2 = (float)((x2 >> 8) | 1u) * 0x1p-24f, u3 = (float)((x3 >> 8) | 1u) * 0x1p-24f;
  const float ra = sqrtf(-2.0f * gh::glog(u0, gh::c_logtab)), rb = sqrtf(-2.0f * gh::glog(u2, gh::c_logtab));
  float sa, ca, sb, cb;
  gh::gsincos(6.28318530717958647692f * u1, sa, ca);
  gh::gsincos(6.28318530717958647692f * u3, sb, cb);
  g[0] = ra * ca;
  g[1] = ra * sa;
  g[2] = rb * cb;
  g[3] = rb * sb;
}

struct Frame {
  float fx, fy, fz, plane_z, ox, oy, oz, weight;
};

// quantile tables (6 x K) and the destination of decoded photons
struct Decode {
  const float *qtab;
  int K;
  float scale, g_max;  // scale = (K - 1) / (2 g_max)
  Frame f;
  float *out[8];
};

__device__ __forceinline__ float qdecode(const float *__restrict__ q, int K, float scale, float g_max, float g) {
  float t = (g + g_max) * scale;
  t = fminf(fmaxf(t, 0.0f), (float)(K - 1));  // NaN -> 0
  const int k = min((int)t, K - 2);
  const float a = t - (float)k;
  const float q0 = q[k], q1 = q[k + 1];
  return fmaf(a, q1 - q0, q0);
}

// photon i from the generator's 6 outputs z
__device__ __forceinline__ void decode(const Decode &d, int64_t i, const float (&z)[6]) {
  const int K = d.K;
  const Frame &f = d.f;
  const float E = qdecode(d.qtab, K, d.scale, d.g_max, z[0]);
  const float px = qdecode(d.qtab + K, K, d.scale, d.g_max, z[1]);
  const float py = qdecode(d.qtab + 2 * K, K, d.scale, d.g_max, z[2]);
  float lu = qdecode(d.qtab + 3 * K, K, d.scale, d.g_max, z[3]);
  float lv = qdecode(d.qtab + 4 * K, K, d.scale, d.g_max, z[4]);
  float lw = qdecode(d.qtab + 5 * K, K, d.scale, d.g_max, z[5]);
  const float l2 = fmaf(lw, lw, fmaf(lv, lv, lu * lu));
  if (!(l2 > 0.0f)) { lu = 0.0f; lv = 0.0f; lw = 1.0f; }
  else gh::normalize3(lu, lv, lw);
  float nx = px - f.fx, ny = py - f.fy, nz = f.plane_z - f.fz;
  gh::normalize3(nx, ny, nz);
  const float up = sqrtf(fmaf(ny, ny, nx * nx));
  float e1x, e1y, e1z, e2x, e2y;
  if (up > 1e-7f) {
    const float iu = 1.0f / up;
    e1x = (nx * nz) * iu; e1y = (ny * nz) * iu; e1z = -up;
    e2x = -ny * iu; e2y = nx * iu;
  } else {
    e1x = nz; e1y = 0.0f; e1z = 0.0f;
    e2x = 0.0f; e2y = 1.0f;
  }
  float du = fmaf(lw, nx, fmaf(lv, e2x, lu * e1x));
  float dv = fmaf(lw, ny, fmaf(lv, e2y, lu * e1y));
  float dw = fmaf(lw, nz, lu * e1z);
  gh::normalize3(du, dv, dw);
  d.out[0][i] = px + f.ox; d.out[1][i] = py + f.oy; d.out[2][i] = f.plane_z + f.oz;
  d.out[3][i] = du; d.out[4][i] = dv; d.out[5][i] = dw;
  d.out[6][i] = E; d.out[7][i] = f.weight;
}

}  // namespace ep
