// Training losses of the learned models, each with its gradient in one launch.
//
// gh_sliced_w2: sliced 2-Wasserstein loss of two sets of M points (rows of K values) on P
// projections. A projection is one 1-D optimal transport problem: with both sets' projected
// values sorted, loss = mean (a_(i) - b_(i))^2 and dloss/da of the element that sorts to
// position i is 2 (a_(i) - b_(i)) / (M P). One 1024-thread workgroup per projection projects
// and sorts both sets in its LDS: only the points are read and the gradient written. The
// library form (two products, two segmented sorts with index arrays, the differences, squares
// and their gradients, a scatter; some 25 launches) took 640 us at 16384 x 134, this one 113
// (8 the projections, 94 the sorts, 7 the gradient's transposition; 36 us at 1024 rows). It is
// bound by the digit ranking of its eight radix passes, on one CU per projection.
//
// Sort: least-significant-digit radix, 4 passes of 8 bits over the order-preserving integer of
// the FP32 value, stable, so equal values keep their index order. Wave w holds elements
// 64 w E + 64 r + lane (E per thread) in registers; a pass ranks them round by round with 8
// ballots (the lanes of a round with the same digit) on per-wave digit counters, scans the
// counters (digit-major), and scatters through LDS. 16384 keys and 16-bit indices and the
// counters take 112 KiB. (With the lanes of equal digits found by 64-bit selects instead of the
// 3-input operation: 180 us; with the gradient written in place, 4-byte values 4 P apart: 128.)
//
// gh_softmax_ce: mean softmax cross-entropy and its gradient for logits of few classes in one
// launch of 4.5 us (5003 x 4); the library form took 12 launches, 45 us and more on the host.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/gatehip.h"

namespace {

constexpr int W2_THREADS = 1024, W2_WAVES = W2_THREADS / 64;

__device__ __forceinline__ uint32_t sort_key(float x) {
  if (x != x) return 0xFFFFFFFFu;  // NaN last
  const uint32_t u = __float_as_uint(x + 0.0f);  // -0 and 0 are equal
  return u ^ ((u >> 31) ? 0xFFFFFFFFu : 0x80000000u);
}
__device__ __forceinline__ float sort_value(uint32_t k) {
  return __uint_as_float(k ^ ((k >> 31) ? 0x80000000u : 0xFFFFFFFFu));
}

// inclusive scan over the wave in 6 cross-lane adds (row shifts, then row broadcasts)
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
#define GH_DPP_ADD(CTRL, ROWS) \
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false)
  GH_DPP_ADD(0x111, 0xF);  // row_shr:1
  GH_DPP_ADD(0x112, 0xF);  // row_shr:2
  GH_DPP_ADD(0x114, 0xF);  // row_shr:4
  GH_DPP_ADD(0x118, 0xF);  // row_shr:8
  GH_DPP_ADD(0x142, 0xA);  // row_bcast:15 into rows 1 and 3
  GH_DPP_ADD(0x143, 0xC);  // row_bcast:31 into rows 2 and 3
#undef GH_DPP_ADD
  return v;
}

// Stable sort of the workgroup's 1024 E (key, index) pairs; on return thread (wave w, lane)
// holds positions 64 w E + 64 r + lane. cnt: [wave][256], zero on entry and on return; part:
// [4][256], tot: [4].
template <int E, bool INDEX>
__device__ __forceinline__ void radix_sort(uint32_t (&key)[E], uint32_t (&idx)[E], uint32_t *s_key, uint16_t *s_idx,
                                           uint32_t *cnt, uint32_t *part, uint32_t *tot) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  volatile uint32_t *mine = cnt + wave * 256;
  for (int shift = 0; shift < 32; shift += 8) {
    // (the rank, below 1024 E <= 2^14, goes into the index register's upper half)
#pragma unroll
    for (int r = 0; r < E; ++r) {
      // lanes of this round with the same digit: per bit, one compare and two 3-input operations
      uint32_t lo = ~0u, hi = ~0u;
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const uint32_t bit = (uint32_t)__builtin_amdgcn_sbfe((int)key[r], shift + b, 1);  // 0 or ~0
        const uint64_t set = __ballot(bit != 0u);
        lo = __builtin_amdgcn_bitop3_b32(lo, (uint32_t)set, bit, 0x90);  // lo & ~(set ^ bit)
        hi = __builtin_amdgcn_bitop3_b32(hi, (uint32_t)(set >> 32), bit, 0x90);
      }
      const uint32_t d = (key[r] >> shift) & 255u;
      const uint32_t before = mine[d];
      const uint32_t ahead = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
      idx[r] = (idx[r] & 0xFFFFu) | (before + ahead) << 16;
      // the wave's LDS operations complete in order: the next round reads the new count
      if (ahead == 0u) mine[d] = before + (uint32_t)(__popc(lo) + __popc(hi));
      // (the scheduler would hoist the ballots of every round, whose masks do not fit in registers)
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    {
      // exclusive scan of the counters, digit-major: thread (digit d, quarter q of the waves);
      // every quarter scans the 256 digit totals for itself
      const int d = tid & 255, q = tid >> 8;
      uint32_t c[4], sum = 0u;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        c[k] = cnt[(4 * q + k) * 256 + d];
        sum += c[k];
      }
      part[q * 256 + d] = sum;
      __syncthreads();
      uint32_t all = 0u, off = 0u;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t v = part[k * 256 + d];
        off += k < q ? v : 0u;
        all += v;
      }
      const uint32_t inc = wave_scan(all);
      if (q == 0 && lane == 63) tot[wave] = inc;
      __syncthreads();
      uint32_t base = inc - all + off;
#pragma unroll
      for (int k = 0; k < 3; ++k) base += k < (d >> 6) ? tot[k] : 0u;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        cnt[(4 * q + k) * 256 + d] = base;
        base += c[k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const uint32_t at = mine[(key[r] >> shift) & 255u] + (idx[r] >> 16);
      s_key[at] = key[r];
      if (INDEX) s_idx[at] = (uint16_t)idx[r];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) mine[lane + k * 64] = 0u;  // this wave is done with its counters
    __syncthreads();
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const int at = (wave * E + r) * 64 + lane;
      key[r] = s_key[at];
      idx[r] = INDEX ? s_idx[at] : 0u;
    }
  }
}

constexpr int W2_MAX_K = 8, W2_COLS = 32;
struct W2Args {
  const float *A, *B, *dir;  // M x K (pitches lda, ldb), M x K, K x P
  int64_t lda, ldb;
  int M, K, P;
  float scale;               // 1 / (M P)
  float *a, *b;              // projections, P x M; the gradient takes a's place
  float *grad, *loss;        // M x P, P
};

// projections of both sets, one set per blockIdx.z, W2_COLS columns per blockIdx.y: a row of
// points is read once for them, and the values leave column by column in row order, so that the
// sorting workgroups read whole lines (read in place, M x P row-major, or projected there from
// the 24-byte rows, the columns took 25-50 us)
__global__ void __launch_bounds__(256) w2_project_kernel(W2Args w) {
  __shared__ float s_dir[W2_COLS][W2_MAX_K];
  const int c0 = blockIdx.y * W2_COLS, n = min(W2_COLS, w.P - c0);
  {
    const int c = threadIdx.x / W2_MAX_K, k = threadIdx.x % W2_MAX_K;
    static_assert(W2_COLS * W2_MAX_K == 256, "one direction value per thread");
    s_dir[c][k] = c < n && k < w.K ? w.dir[k * w.P + c0 + c] : 0.0f;
  }
  __syncthreads();
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= w.M) return;
  const float *row = blockIdx.z ? w.B + i * w.ldb : w.A + i * w.lda;
  float *out = (blockIdx.z ? w.b : w.a) + (int64_t)c0 * w.M + i;
  float x[W2_MAX_K];
#pragma unroll
  for (int k = 0; k < W2_MAX_K; ++k) x[k] = k < w.K ? row[k] : 0.0f;
#pragma unroll 4
  for (int c = 0; c < n; ++c) {
    float v = 0.0f;
#pragma unroll
    for (int k = 0; k < W2_MAX_K; ++k) {
      const float p = fmaf(x[k], s_dir[c][k], v);
      v = k < w.K ? p : v;
    }
    out[(int64_t)c * w.M] = v;
  }
}

template <int E>
__global__ void __launch_bounds__(W2_THREADS) sliced_w2_kernel(W2Args w) {
  extern __shared__ __align__(16) unsigned char w2_lds[];
  uint32_t *s_key = (uint32_t *)w2_lds;
  uint32_t *cnt = s_key + W2_THREADS * E;
  uint32_t *part = cnt + W2_WAVES * 256;
  uint32_t *tot = part + 4 * 256;
  uint16_t *s_idx = (uint16_t *)(tot + 8);
  const int col = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t key[E], idx[E];
  float b[E];
  // element r of the thread: row i0 + 64 r
  const int i0 = wave * E * 64 + lane;
  auto load = [&](const float *src) {
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const int i = i0 + r * 64;
      key[r] = i < w.M ? sort_key(src[i]) : 0xFFFFFFFFu;
      idx[r] = (uint32_t)i;
    }
  };
#pragma unroll
  for (int k = 0; k < 4; ++k) cnt[threadIdx.x + k * W2_THREADS] = 0u;
  __syncthreads();
  load(w.b + (int64_t)col * w.M);
  radix_sort<E, false>(key, idx, s_key, s_idx, cnt, part, tot);
#pragma unroll
  for (int r = 0; r < E; ++r) b[r] = sort_value(key[r]);
  load(w.a + (int64_t)col * w.M);
  radix_sort<E, true>(key, idx, s_key, s_idx, cnt, part, tot);
  float sum = 0.0f;
  __syncthreads();  // every wave has read its sorted keys
  float *s_grad = (float *)s_key;
#pragma unroll
  for (int r = 0; r < E; ++r) {
    if (i0 + r * 64 < w.M) {
      const float x = sort_value(key[r]) - b[r];
      sum = fmaf(x, x, sum);
      s_grad[idx[r]] = w.scale * (2.0f * x);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  float *s_sum = (float *)part;
  if (lane == 0) s_sum[wave] = sum;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int i = r * W2_THREADS + (int)threadIdx.x;
    if (i < w.M) w.a[(int64_t)col * w.M + i] = s_grad[i];
  }
  if (threadIdx.x == 0) {
    float s = 0.0f;
    for (int k = 0; k < W2_WAVES; ++k) s += s_sum[k];
    w.loss[col] = s;
  }
}

// the gradient from P x M to M x P, in tiles of 64 x 64 through LDS (each workgroup writing its
// column of 4-byte values 4 P bytes apart took 30 us at 16384 x 134)
__global__ void __launch_bounds__(256) w2_transpose_kernel(W2Args w) {
  __shared__ float t[64][65];
  const int i0 = blockIdx.x * 64, c0 = blockIdx.y * 64, x = threadIdx.x & 63, y = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < 64; k += 4)
    if (c0 + k + y < w.P && i0 + x < w.M) t[k + y][x] = w.a[(int64_t)(c0 + k + y) * w.M + i0 + x];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 64; k += 4)
    if (i0 + k + y < w.M && c0 + x < w.P) w.grad[(int64_t)(i0 + k + y) * w.P + c0 + x] = t[x][k + y];
}

template <int E>
int launch_w2(const W2Args &w, hipStream_t st) {
  const size_t lds = (size_t)W2_THREADS * E * 6 + (W2_WAVES + 4) * 256 * 4 + 32;
  const void *fn = (const void *)&sliced_w2_kernel<E>;
  if (lds > 64 * 1024 && hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return GH_EHIP;
  hipLaunchKernelGGL(w2_project_kernel, dim3((w.M + 255) / 256, (w.P + W2_COLS - 1) / W2_COLS, 2), dim3(256), 0, st, w);
  if (hipGetLastError() != hipSuccess) return GH_EHIP;
  hipLaunchKernelGGL(sliced_w2_kernel<E>, dim3(w.P), dim3(W2_THREADS), lds, st, w);
  if (hipGetLastError() != hipSuccess) return GH_EHIP;
  hipLaunchKernelGGL(w2_transpose_kernel, dim3((w.M + 63) / 64, (w.P + 63) / 64), dim3(256), 0, st, w);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}

constexpr int CE_MAX_CLASSES = 16;

// one row per thread; loss[block] = sum over the block's rows of -log p(class)
__global__ void __launch_bounds__(256) softmax_ce_kernel(const float *__restrict__ Z, int64_t ldz, int M, int C,
                                                         const int64_t *__restrict__ cls, const int64_t *__restrict__ rows,
                                                         float *__restrict__ grad, float *__restrict__ loss) {
  __shared__ float s_sum[4];
  const int i = blockIdx.x * 256 + threadIdx.x;
  float l = 0.0f;
  if (i < M) {
    const float *z = Z + i * ldz;
    const int y = (int)cls[rows ? rows[i] : i];
    float v[CE_MAX_CLASSES], e[CE_MAX_CLASSES], mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < CE_MAX_CLASSES; ++k)
      if (k < C) { v[k] = z[k]; mx = fmaxf(mx, v[k]); }
#pragma unroll
    for (int k = 0; k < CE_MAX_CLASSES; ++k) e[k] = k < C ? expf(v[k] - mx) : 0.0f;
    // halves added onto halves, as a reduction over lanes adds them
#pragma unroll
    for (int o = CE_MAX_CLASSES / 2; o > 0; o >>= 1)
#pragma unroll
      for (int k = 0; k < o; ++k) e[k] += e[k + o];
    const float lse = logf(e[0]), scale = 1.0f / (float)M;
#pragma unroll
    for (int k = 0; k < CE_MAX_CLASSES; ++k)
      if (k < C) {
        const float lp = (v[k] - mx) - lse;
        if (k == y) l = -lp;
        grad[(int64_t)i * C + k] = (expf(lp) - (k == y ? 1.0f : 0.0f)) * scale;
      }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
  if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = l;
  __syncthreads();
  if (threadIdx.x == 0) loss[blockIdx.x] = (s_sum[0] + s_sum[1]) + (s_sum[2] + s_sum[3]);
}

}  // namespace

extern "C" int gh_sliced_w2(const float *A, int64_t lda, const float *B, int64_t ldb, const float *dir, int32_t M,
                            int32_t K, int32_t P, float *work, float *grad, float *loss, void *stream) {
  if (!A || !B || !dir || !work || !grad || !loss || M <= 0 || M > GH_SLICED_W2_MAX_ROWS || K <= 0 || K > W2_MAX_K || lda < K ||
      ldb < K || P <= 0 || (int64_t)M * P > INT32_MAX)
    return GH_EINVAL;
  const W2Args w{A, B, dir, lda, ldb, M, K, P, 1.0f / (float)((double)M * (double)P),
                 work, work + (int64_t)M * P, grad, loss};
  hipStream_t st = (hipStream_t)stream;
  if (M <= 4 * W2_THREADS) return launch_w2<4>(w, st);
  if (M <= 8 * W2_THREADS) return launch_w2<8>(w, st);
  return launch_w2<16>(w, st);
}

extern "C" int gh_softmax_ce(const float *Z, int64_t ldz, int32_t M, int32_t n_classes, const int64_t *cls,
                             const int64_t *rows, float *grad, float *loss, void *stream) {
  if (!Z || !cls || !grad || !loss || M <= 0 || n_classes <= 0 || n_classes > CE_MAX_CLASSES || ldz < n_classes)
    return GH_EINVAL;
  hipLaunchKernelGGL(softmax_ce_kernel, dim3((M + 255) / 256), dim3(256), 0, (hipStream_t)stream, Z, ldz, (int)M,
                     (int)n_classes, cls, rows, grad, loss);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}
