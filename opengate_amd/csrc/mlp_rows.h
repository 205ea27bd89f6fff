// Row-tile form of the dense network: one workgroup of 8 waves carries 16 RT rows through every
// layer. Shared by inference on few rows (mlp.hip) and by the training passes (mlp_train.hip).
//
// What bounds it: a batch of 1e3..4e4 rows gives every CU one tile of 16..64 rows, so a layer
// lasts 1-4 us and its weights (H x H bf16, 128 KiB at H = 256) come from L2 in that time. The
// waves form CG column groups x 8 / CG row groups; at H = 256 (CG = 8) each owns 32 output
// columns for all rows of the tile, so no two waves of a workgroup read the same weights. A
// wave holds its weights as MFMA fragments in registers; those of the next layer are loaded
// into them as this layer's steps are done with them. One barrier per layer. The
// activations go through LDS in fragment order: 16-byte unit (row tile i, k step ks, lane l) at
// ((i NK + ks) 64 + l) 16, lane l holding row l % 16 and k = 32 ks + 8 (l / 16) + 0..7, so the
// reads and writes of a wave are consecutive (no bank conflicts). Two activation buffers
// alternate. The MFMA sequence of an output element (k steps of 32 in order, bias, ReLU, bf16
// rounding) is that of the layer-by-layer GEMMs: bit-identical results.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#include "exitplane.h"

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
  const __bf16 *wt[MAXL];   // [N_l][K_l], rows of K_l values or fragment order
  const float *bias[MAXL];  // [N_l]
  int n_layers;
  int k_in;                 // valid input columns (<= K0)
  int n_out;                // valid output columns (<= NOUT)
  int x_vec;                // 1: input rows 16-byte aligned (16-byte loads)
};

// What the backward pass needs, in tiles of 16 rows, each in the fragment order of the
// activation buffer (a wave's store is 512 consecutive bytes), padded to a multiple of 32 rows
// with zeros: the network's input (32 columns) and each hidden layer's output (H columns)
struct MlpKeep {
  __bf16 *x;
  __bf16 *y[MAXL];
};
// The exit-plane generator in one launch: the input rows are noise rows first .. first + M - 1
// (n_cols columns), the output rows are decoded into photons
struct MlpGenerate {
  uint32_t k0, k1;
  uint64_t first;
  int n_cols;
  ep::Decode d;
};

// 8 noise columns 8 unit .. of row `row` as a 16-byte unit of the input tile
__device__ __forceinline__ bf16x8 noise_unit(const MlpGenerate &gen, uint64_t row, int unit) {
  bf16x8 v = bf16x8_zero();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = 8 * unit + 4 * h;
    if (c >= gen.n_cols) break;
    float g[4];
    ep::noise4(row, (uint32_t)(c >> 2), gen.k0, gen.k1, g);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (c + j < gen.n_cols) v[4 * h + j] = (__bf16)g[j];
  }
  return v;
}

enum { ROWS_INFER = 0, ROWS_KEEP = 1, ROWS_GENERATE = 2 };

__host__ __device__ inline int64_t padded_rows(int64_t M) { return (M + 31) & ~(int64_t)31; }

// workgroups of 16 RT rows that cover the padded rows
inline int64_t row_grid(int64_t M, int RT) { return (padded_rows(M) + 16 * RT - 1) / (16 * RT); }

// rows of a tile for M rows: the smallest tile that still gives each of 256 CUs at most one
inline int row_tiles(int64_t M) { return M <= 16 * 256 ? 1 : (M <= 32 * 256 ? 2 : 4); }

// two activation buffers
template <int H, int RT>
constexpr size_t rows_lds_bytes() { return 2ull * 16 * RT * H * sizeof(__bf16); }

// MFMAs of one layer of K = 32 NK: acc += W (A operand, fragments w) x activations (B operand).
// A fragment's registers are free after its step: `next` (the same wave's column tiles of the
// next layer, lane offset included, `step` elements from tile to tile) is loaded into them.
template <int RT, int CT, int NK>
__device__ __forceinline__ void rows_mma(floatx4 (&acc)[RT][CT], bf16x8 (&w)[NK][CT], const __bf16 *in, int lane,
                                         const __bf16 *next, int step) {
#pragma unroll
  for (int ks = 0; ks < NK; ++ks) {
    bf16x8 af[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) af[i] = *(const bf16x8 *)(in + ((i * NK + ks) * 64 + lane) * 8);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[ks][j], af[i], acc[i][j], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < CT; ++j) w[ks][j] = *(const bf16x8 *)(next + j * step + ks * 512);
  }
}

// the first layer's single step (K = 32); its activation tile has the pitch of NK steps
template <int RT, int CT, int NK>
__device__ __forceinline__ void rows_mma0(floatx4 (&acc)[RT][CT], const bf16x8 (&w)[CT], const __bf16 *in, int lane) {
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const bf16x8 af = *(const bf16x8 *)(in + (i * NK * 64 + lane) * 8);
#pragma unroll
    for (int j = 0; j < CT; ++j)
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], af, acc[i][j], 0, 0, 0);
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

// fragments of CT column tiles of a weight matrix in fragment order, K = 32 NK: 1 KiB per
// fragment, read by the 64 lanes in one piece. W: the first tile with the lane's offset, `step`
// elements from tile to tile. (Read from rows of K values instead, a fragment is 16 pieces of
// 64 bytes: 3.4 us for the 128 KiB of a layer against 1.0 us; the six-layer forward of 1000
// rows 19.6 -> 8.3 us, of 16384 rows 20.3 -> 12.0.)
template <int CT, int NK>
__device__ __forceinline__ void rows_weights(bf16x8 (&w)[NK][CT], const __bf16 *W, int step) {
#pragma unroll
  for (int ks = 0; ks < NK; ++ks)
#pragma unroll
    for (int j = 0; j < CT; ++j) w[ks][j] = *(const bf16x8 *)(W + j * step + ks * 512);
}

// Forward through all layers. MODE: inference (Z: columns 0..n_out-1), training (also keeps the
// activations), or noise -> photons (X and Z unused).
template <int H, int RT, int CG, int MODE>
__global__ void __launch_bounds__(ROW_THREADS) mlp_rows_forward(const __bf16 *__restrict__ X, int64_t ldx, int64_t M,
                                                                MlpArgs a, MlpKeep keep, MlpGenerate gen,
                                                                float *__restrict__ Z, int64_t ldz) {
  constexpr bool KEEP = MODE == ROWS_KEEP, GENERATE = MODE == ROWS_GENERATE;
  // RW row tiles and CT column tiles per wave. (CG is 8 everywhere; with the row offset i0, then
  // zero, folded away, the training forward at 16384 rows takes 19.4 us instead of 18.7: the
  // addresses in registers leave the compiler a better order.)
  constexpr int NK = H / 32, RG = 8 / CG, CT = H / 16 / CG, RW = RT / RG, ROWS = 16 * RT;
  static_assert(RT % RG == 0, "the row groups share the tile's row tiles evenly");
  extern __shared__ __align__(16) unsigned char mlp_lds[];
  __bf16 *in = (__bf16 *)mlp_lds, *out = in + ROWS * H;
  float *s_bias = (float *)(mlp_lds + 2 * ROWS * H * sizeof(__bf16));  // [layer][H]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, g = lane >> 4;
  const int cg = wave % CG, i0 = wave / CG * RW;
  const int n0 = cg * 16 * CT;
  const int64_t row0 = (int64_t)blockIdx.x * ROWS;
  const int L = a.n_layers;
  bf16x8 w0[CT], w[NK][CT];
  // weights of layer l >= 1: a hidden layer's column tiles, or the output layer's 16 columns
  // (past the end: the output layer again; a branch around the loads would make the compiler
  // wait for all of them in the path without)
  auto tiles = [&](int l) { return a.wt[min(l, L - 1)] + (l < L - 1 ? cg * CT * NK * 512 : 0) + lane * 8; };
  auto step = [&](int l) { return l < L - 1 ? NK * 512 : 0; };
#pragma unroll
  for (int j = 0; j < CT; ++j) w0[j] = *(const bf16x8 *)(a.wt[0] + ((cg * CT + j) * 64 + lane) * 8);
  for (int u = tid; u < ROWS * 4; u += ROW_THREADS) {
    const int r = u >> 2, q = (u & 3) * 8;
    const int64_t gr = row0 + r;
    bf16x8 v = bf16x8_zero();
    if (GENERATE) {
      if (gr < M && q < gen.n_cols) v = noise_unit(gen, gen.first + (uint64_t)gr, u & 3);
    } else if (gr < M && q < a.k_in) {
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
    if (KEEP && gr < padded_rows(M))
      *(bf16x8 *)(keep.x + row0 * K0 + ((r >> 4) * 64 + (u & 3) * 16 + (r & 15)) * 8) = v;
  }
  // biases in LDS: a bias load behind the next layer's weights would wait for all of them
  // (loads return in order)
  for (int u = tid; u < (L - 1) * (H / 4); u += ROW_THREADS)
    ((floatx4 *)s_bias)[u] = ((const floatx4 *)a.bias[u / (H / 4)])[u % (H / 4)];
  rows_weights<CT, NK>(w, tiles(1), step(1));
  __syncthreads();
  floatx4 acc[RW][CT];
  // bias, ReLU, bf16; into the other activation buffer and, in training, to memory
  auto finish = [&](int l) {
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int c = n0 + j * 16 + g * 4;
      const floatx4 b = *(const floatx4 *)(s_bias + l * H + c);
#pragma unroll
      for (int i = 0; i < RW; ++i) {
        bf16x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (__bf16)fmaxf(acc[i][j][r] + b[r], 0.0f);
        *(bf16x4 *)(out + rows_at<NK>(i0 + i, fr, c)) = v;
        if (KEEP) {
          const int64_t row = row0 + (i0 + i) * 16 + fr;
          if (row >= M)
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = (__bf16)0.0f;
          if (row < padded_rows(M)) *(bf16x4 *)(keep.y[l] + row0 * H + rows_at<NK>(i0 + i, fr, c)) = v;
        }
      }
    }
    __syncthreads();
    __bf16 *t = in; in = out; out = t;
  };
  rows_zero<RW, CT>(acc);
  rows_mma0<RW, CT, NK>(acc, w0, in + i0 * NK * 512, lane);
  finish(0);
  for (int l = 1; l < L - 1; ++l) {
    rows_zero<RW, CT>(acc);
    rows_mma<RW, CT, NK>(acc, w, in + i0 * NK * 512, lane, tiles(l + 1), step(l + 1));
    finish(l);
  }
  // output layer: row tiles wave, wave + 8, ...
  for (int i = wave; i < RT; i += 8) {
    floatx4 o = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      const bf16x8 af = *(const bf16x8 *)(in + ((i * NK + ks) * 64 + lane) * 8);
      o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, w[ks][0], o, 0, 0, 0);
    }
    if (fr < a.n_out) {
      const float b = a.bias[L - 1][fr];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = row0 + i * 16 + g * 4 + r;
        if (GENERATE) s_bias[(i * 16 + g * 4 + r) * 8 + fr] = o[r] + b;  // (the biases are done with)
        else if (row < M) Z[row * ldz + fr] = o[r] + b;
      }
    }
  }
  if (GENERATE) {
    __syncthreads();
    const int64_t row = row0 + tid;
    if (tid < ROWS && row < M) {
      float z[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) z[k] = s_bias[tid * 8 + k];
      ep::decode(gen.d, row, z);
    }
  }
}

template <int H, int RT, int CG, int MODE>
int launch_rows_forward(const __bf16 *X, int64_t ldx, int64_t M, const MlpArgs &a, const MlpKeep &keep,
                        const MlpGenerate &gen, float *Z, int64_t ldz, hipStream_t st) {
  size_t extra = (a.n_layers - 1) * H * sizeof(float);
  if (MODE == ROWS_GENERATE) extra = extra > 16 * RT * 8 * sizeof(float) ? extra : 16 * RT * 8 * sizeof(float);
  const size_t lds = rows_lds_bytes<H, RT>() + extra;
  const void *fn = (const void *)&mlp_rows_forward<H, RT, CG, MODE>;
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return 2;  // GH_EHIP
  const dim3 grid((unsigned)(MODE == ROWS_KEEP ? row_grid(M, RT) : (M + 16 * RT - 1) / (16 * RT)));
  hipLaunchKernelGGL((mlp_rows_forward<H, RT, CG, MODE>), grid, dim3(ROW_THREADS), lds, st, X, ldx, M, a, keep, gen, Z,
                     ldz);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

}  // namespace mlp
