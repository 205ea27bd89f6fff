// Row-tile form of the dense network: one workgroup of 8 waves carries 16 RT rows through every
// layer. Shared by inference on few rows (mlp.hip) and by the training passes (mlp_train.hip).
//
// What bounds it: a batch of 1e3..4e4 rows gives every CU one tile of 16..64 rows, so a layer
// lasts 1-4 us and its weights (H x H bf16, 128 KiB at H = 256) come from L2 in that time. Each
// wave owns H / 8 output columns for all rows of the tile, so no two waves of a workgroup read
// the same weights; it holds them as MFMA fragments in registers, and the next layer's are
// loaded while this layer multiplies (two register sets, one barrier per layer). The
// activations go through LDS in fragment order: 16-byte unit (row tile i, k step ks, lane l) at
// ((i NK + ks) 64 + l) 16, lane l holding row l % 16 and k = 32 ks + 8 (l / 16) + 0..7, so the
// reads and writes of a wave are consecutive (no bank conflicts). Two activation buffers
// alternate. The MFMA sequence of an output element (k steps of 32 in order, bias, ReLU, bf16
// rounding) is that of the layer-by-layer GEMMs: bit-identical results.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

namespace mlp {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int MAXL = 8;   // layers
constexpr int K0 = 32;    // first-layer input width (padded)
constexpr int NOUT = 16;  // last-layer output width (padded)
constexpr int ROW_THREADS = 512;

__device__ __forceinline__ bf16x8 bf16x8_zero() {
  bf16x8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = (__bf16)0.0f;
  return v;
}

struct MlpArgs {
  const __bf16 *wt[MAXL];   // [N_l][K_l]
  const float *bias[MAXL];  // [N_l]
  int n_layers;
  int k_in;                 // valid input columns (<= K0)
  int n_out;                // valid output columns (<= NOUT)
  int x_vec;                // 1: input rows 16-byte aligned (16-byte loads)
};

// hidden activations kept for the backward pass: layer l's output, M x H row-major
struct MlpKeep {
  __bf16 *y[MAXL];
};

// rows of a tile for M rows: the smallest tile that still gives each of 256 CUs at most one
inline int row_tiles(int64_t M) { return M <= 16 * 256 ? 1 : (M <= 32 * 256 ? 2 : 4); }

template <int H, int RT>
constexpr size_t rows_lds_bytes() { return 2ull * 16 * RT * H * sizeof(__bf16); }

// MFMAs of one layer of K = 32 NK: acc += W (A operand, fragments w) x activations (B operand)
template <int RT, int CT, int NK, int NKH, int NW>
__device__ __forceinline__ void rows_mma(floatx4 (&acc)[RT][CT], const bf16x8 (&w)[NW][CT], const __bf16 *in,
                                         int lane) {
#pragma unroll
  for (int ks = 0; ks < NK; ++ks) {
    bf16x8 af[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) af[i] = *(const bf16x8 *)(in + ((i * NKH + ks) * 64 + lane) * 8);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[ks][j], af[i], acc[i][j], 0, 0, 0);
  }
}

template <int RT, int CT>
__device__ __forceinline__ void rows_zero(floatx4 (&acc)[RT][CT]) {
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
}

// element offset of columns c..c+3 (c a multiple of 4) of row 16 i + fr in an activation buffer
template <int NK>
__device__ __forceinline__ int rows_at(int i, int fr, int c) {
  return ((i * NK + (c >> 5)) * 64 + ((c >> 3) & 3) * 16 + fr) * 8 + (c & 4);
}

// fragments of CT column tiles (n0, n0 + step, ...) of a weight matrix [N][K], K = 32 NK contiguous
template <int CT, int NK>
__device__ __forceinline__ void rows_weights(bf16x8 (&w)[NK][CT], const __bf16 *W, int K, int n0, int step, int fr,
                                             int fk) {
#pragma unroll
  for (int ks = 0; ks < NK; ++ks)
#pragma unroll
    for (int j = 0; j < CT; ++j) w[ks][j] = *(const bf16x8 *)(W + (int64_t)(n0 + j * step + fr) * K + ks * 32 + fk);
}

// Forward through all layers; KEEP stores the hidden activations. Z: columns 0..n_out-1.
template <int H, int RT, bool KEEP>
__global__ void __launch_bounds__(ROW_THREADS) mlp_rows_forward(const __bf16 *__restrict__ X, int64_t ldx, int64_t M,
                                                                MlpArgs a, MlpKeep keep, float *__restrict__ Z,
                                                                int64_t ldz) {
  constexpr int NK = H / 32, CT = H / 128, ROWS = 16 * RT;
  extern __shared__ __align__(16) unsigned char mlp_lds[];
  __bf16 *in = (__bf16 *)mlp_lds, *out = in + ROWS * H;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fr = lane & 15, g = lane >> 4, fk = g * 8;
  const int n0 = wave * 16 * CT;
  const int64_t row0 = (int64_t)blockIdx.x * ROWS;
  const int L = a.n_layers;
  bf16x8 w0[1][CT], wA[NK][CT], wB[NK][CT];
  // weights of layer l >= 1: a hidden layer's column tiles, or the output layer's 16 columns
  auto fetch = [&](bf16x8(&w)[NK][CT], int l) {
    if (l < L) rows_weights<CT, NK>(w, a.wt[l], H, l < L - 1 ? n0 : 0, l < L - 1 ? 16 : 0, fr, fk);
    // left alone, the scheduler sinks these loads to their use in the next layer
    __builtin_amdgcn_sched_barrier(0);
  };
  rows_weights<CT, 1>(w0, a.wt[0], K0, n0, 16, fr, fk);
  for (int u = tid; u < ROWS * 4; u += ROW_THREADS) {
    const int r = u >> 2, q = (u & 3) * 8;
    const int64_t gr = row0 + r;
    bf16x8 v = bf16x8_zero();
    if (gr < M && q < a.k_in) {
      if (a.x_vec) {
        v = *(const bf16x8 *)(X + gr * ldx + q);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (q + j >= a.k_in) v[j] = (__bf16)0.0f;
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (q + j < a.k_in) v[j] = X[gr * ldx + q + j];
      }
    }
    *(bf16x8 *)(in + (((r >> 4) * NK) * 64 + (u & 3) * 16 + (r & 15)) * 8) = v;
  }
  fetch(wA, 1);
  __syncthreads();
  floatx4 acc[RT][CT];
  // bias, ReLU, bf16; into the other activation buffer and, in training, to memory
  auto finish = [&](int l) {
    const float *bias = a.bias[l];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int c = n0 + j * 16 + g * 4;
      const floatx4 b = *(const floatx4 *)(bias + c);
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        bf16x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (__bf16)fmaxf(acc[i][j][r] + b[r], 0.0f);
        *(bf16x4 *)(out + rows_at<NK>(i, fr, c)) = v;
        if (KEEP) {
          const int64_t row = row0 + i * 16 + fr;
          if (row < M) *(bf16x4 *)(keep.y[l] + row * H + c) = v;
        }
      }
    }
    __syncthreads();
    __bf16 *t = in; in = out; out = t;
  };
  auto hidden = [&](int l, bf16x8(&w)[NK][CT]) {
    rows_zero<RT, CT>(acc);
    rows_mma<RT, CT, NK, NK, NK>(acc, w, in, lane);
    finish(l);
  };
  // output layer: row tile i by wave i
  auto output = [&](bf16x8(&w)[NK][CT]) {
    if (wave >= RT) return;
    floatx4 o = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      const bf16x8 af = *(const bf16x8 *)(in + ((wave * NK + ks) * 64 + lane) * 8);
      o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, w[ks][0], o, 0, 0, 0);
    }
    if (fr < a.n_out) {
      const float b = a.bias[L - 1][fr];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = row0 + wave * 16 + g * 4 + r;
        if (row < M) Z[row * ldz + fr] = o[r] + b;
      }
    }
  };
  rows_zero<RT, CT>(acc);
  rows_mma<RT, CT, 1, NK, 1>(acc, w0, in, lane);
  finish(0);
  for (int l = 1;; l += 2) {
    if (l == L - 1) { output(wA); break; }
    fetch(wB, l + 1);
    hidden(l, wA);
    if (l + 1 == L - 1) { output(wB); break; }
    fetch(wA, l + 2);
    hidden(l + 1, wB);
  }
}

template <int H, int RT, bool KEEP>
int launch_rows_forward(const __bf16 *X, int64_t ldx, int64_t M, const MlpArgs &a, const MlpKeep &keep, float *Z,
                        int64_t ldz, hipStream_t st) {
  constexpr size_t lds = rows_lds_bytes<H, RT>();
  const dim3 grid((unsigned)((M + 16 * RT - 1) / (16 * RT)));
  hipLaunchKernelGGL((mlp_rows_forward<H, RT, KEEP>), grid, dim3(ROW_THREADS), lds, st, X, ldx, M, a, keep, Z, ldz);
  return hipGetLastError() == hipSuccess ? 0 : 2;  // GH_OK / GH_EHIP
}

}  // namespace mlp
