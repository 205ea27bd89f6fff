// Training passes of a dense network with equal hidden widths (128 or 256) in four launches:
// forward (mlp_rows.h, activations kept), the chain of input gradients with the bias
// gradients' partial sums, every layer's weight gradient, and the sums of their slices. The
// layer-by-layer GEMMs (mlp.hip) need 3 launches a layer and write the FP32 pre-activations
// and gradients that the fused passes keep in registers. Measured for the network
// 8-256x5-6 at 16384 rows: see each kernel.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/gatehip.h"
#include "mlp_rows.h"
#include "splitk.h"

namespace {

using namespace mlp;

typedef short s16x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ input gradients
// G_l = dLoss/dZ_l. G_{L-1} is the caller's; G_{l-1} = (G_l W_l^T) * relu'(Z_{l-1}), the
// derivative taken from the kept activation (bf16(relu(z)) > 0 where z > 0). Same tile, same
// register-held weights as the forward kernel; W_l [K][N] is read as it is (its rows are the
// outputs of this product). The bias gradients are column sums of the FP32 gradients before
// their rounding to bf16: each workgroup writes the sums of its rows.
struct BackArgs {
  const __bf16 *w[MAXL];  // layer l >= 1: [K_l][N_l], N_l contiguous (N of the last layer: np)
  const __bf16 *y[MAXL];  // kept activations
  __bf16 *g[MAXL];        // out: G_l for l <= L-2, M x H
  __bf16 *g_out;          // out: bf16(G_{L-1}), M x 16, zeros from n_out on
  float *g32[MAXL];       // out, optional: the FP32 gradients of the hidden layers, M x H
  float *db;              // out: [workgroup][(L-1) H + 16] partial sums (layer 0 first)
  int n_layers, n_out, np;
};

template <int H, int RT>
__global__ void __launch_bounds__(ROW_THREADS) mlp_rows_backward(const float *__restrict__ G, int64_t ldg, int64_t M,
                                                                 BackArgs a) {
  constexpr int NK = H / 32, CT = H / 128, ROWS = 16 * RT;
  extern __shared__ __align__(16) unsigned char mlp_lds[];
  __shared__ float s_last[ROW_THREADS / 64][NOUT];
  __bf16 *in = (__bf16 *)mlp_lds, *out = in + ROWS * H;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fr = lane & 15, g = lane >> 4, fk = g * 8;
  const int n0 = wave * 16 * CT;
  const int64_t row0 = (int64_t)blockIdx.x * ROWS;
  const int L = a.n_layers;
  float *db = a.db + (int64_t)blockIdx.x * ((L - 1) * H + NOUT);
  bf16x8 w0[1][CT], wA[NK][CT], wB[NK][CT];
#pragma unroll
  for (int j = 0; j < CT; ++j)
    w0[0][j] = fk < a.np ? *(const bf16x8 *)(a.w[L - 1] + (int64_t)(n0 + j * 16 + fr) * a.np + fk) : bf16x8_zero();
  // output gradient tile: bf16, padded to 32 columns
  for (int u = tid; u < ROWS * 4; u += ROW_THREADS) {
    const int r = u >> 2, q = (u & 3) * 8;
    const int64_t gr = row0 + r;
    bf16x8 v = bf16x8_zero();
    if (gr < M && q < NOUT) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (q + j < a.n_out) v[j] = (__bf16)G[gr * ldg + q + j];
      *(bf16x8 *)(a.g_out + gr * NOUT + q) = v;
    }
    *(bf16x8 *)(in + (((r >> 4) * NK) * 64 + (u & 3) * 16 + (r & 15)) * 8) = v;
  }
  {
    // its column sums: thread (row tid / 16, column tid % 16), then lanes, then waves
    float s = 0.0f;
    for (int r = tid >> 4; r < ROWS; r += ROW_THREADS / 16)
      if (row0 + r < M && fr < a.n_out) s += G[(row0 + r) * ldg + fr];
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    if (g == 0) s_last[wave][fr] = s;
  }
  floatx4 acc[RT][CT];
  bf16x4 y[RT][CT];
  auto fetch_w = [&](bf16x8(&w)[NK][CT], int l) {
    if (l >= 1) rows_weights<CT, NK>(w, a.w[l], H, n0, 16, fr, fk);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto fetch_y = [&](int l) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        const int64_t row = row0 + i * 16 + fr;
#pragma unroll
        for (int r = 0; r < 4; ++r) y[i][j][r] = (__bf16)0.0f;
        if (row < M) y[i][j] = *(const bf16x4 *)(a.y[l] + row * H + n0 + j * 16 + g * 4);
      }
  };
  // times the ReLU derivative; column sums; bf16 to the other buffer and to memory
  auto finish = [&](int l) {
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int c = n0 + j * 16 + g * 4;
      floatx4 s = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        bf16x4 v;
        floatx4 z;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          z[r] = acc[i][j][r] * ((float)y[i][j][r] > 0.0f ? 1.0f : 0.0f);
          s[r] += z[r];
          v[r] = (__bf16)z[r];
        }
        *(bf16x4 *)(out + rows_at<NK>(i, fr, c)) = v;
        const int64_t row = row0 + i * 16 + fr;
        if (row < M) {
          *(bf16x4 *)(a.g[l] + row * H + c) = v;
          if (a.g32[l]) *(floatx4 *)(a.g32[l] + row * H + c) = z;
        }
      }
#pragma unroll
      for (int o = 1; o < 16; o <<= 1)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] += __shfl_xor(s[r], o, 64);
      if (fr == 0) *(floatx4 *)(db + l * H + c) = s;
    }
    __syncthreads();
    __bf16 *t = in; in = out; out = t;
  };
  auto hidden = [&](int l, bf16x8(&w)[NK][CT]) {  // G_{l-1} from G_l
    rows_zero<RT, CT>(acc);
    rows_mma<RT, CT, NK, NK, NK>(acc, w, in, lane);
    finish(l - 1);
  };
  fetch_y(L - 2);
  fetch_w(wA, L - 2);
  __syncthreads();
  if (tid < NOUT) {
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < ROW_THREADS / 64; ++k) s += s_last[k][tid];
    db[(L - 1) * H + tid] = s;
  }
  rows_zero<RT, CT>(acc);
  rows_mma<RT, CT, 1, NK, 1>(acc, w0, in, lane);
  finish(L - 2);
  for (int l = L - 2; l >= 1; l -= 2) {
    fetch_y(l - 1);
    fetch_w(wB, l - 1);
    hidden(l, wA);
    if (l == 1) break;
    fetch_y(l - 2);
    fetch_w(wA, l - 2);
    hidden(l - 1, wB);
  }
}

// ------------------------------------------------------------------ weight gradients
// dW_l = X_l^T G_l: reductions over the batch of two row-major matrices. All layers in one
// launch: blockIdx.x is an output tile of some layer, blockIdx.y a slice of the rows. The slices
// are those of gh_gemm_bf16 for the same product (its rule: 512 rows from 2048 rows on, 32
// slices and 256 workgroups for the four inner layers at 16384 rows), so the sums have the
// same bits. 32 rows
// of both operands are staged in LDS per step, loaded into registers one step ahead; the
// fragments (8 consecutive rows of one column) are read with the transposing LDS read
// (ds_read_b64_tr_b16: lane s of 16 names 4 columns of row s / 4, lane i receives 4 rows of
// column i), with the 32-byte chunks of a row XOR-swizzled so that the 8 rows of a half wave
// fall into different banks.
struct DwLayer {
  const __bf16 *A, *B;  // X_l (M x ka, pitch lda) and G_l (M x nb, pitch ldb)
  int lda, ldb, ka, nb;
  int rows, slices;     // rows of a slice, number of slices
  float *part;          // [slice][ka nb] partial sums
  int64_t off;          // offset of the layer's ka x nb block in the result
};
struct DwArgs {
  DwLayer layer[MAXL];
  int n_layers;
  int64_t M, n_elems;   // elements of the result
};

constexpr int DW_THREADS = 512;

__device__ __forceinline__ int dw_swizzle(int row, int units) {
  return (((row & 3) | ((row >> 1) & 4)) << 1) & (units - 1);
}

// output tile [a0, a0 + TA) x [0, TB) over the waves WA x WB
template <int TA, int TB, int WA, int WB>
__device__ __forceinline__ void dw_tile(const DwLayer &d, int a0, int64_t r0, int64_t r1, float *part,
                                        unsigned char *lds) {
  constexpr int UA = TA / 8, UB = TB / 8, UNITS = 32 * (UA + UB), NU = (UNITS + DW_THREADS - 1) / DW_THREADS;
  constexpr int FA = TA / 16 / WA, FB = TB / 16 / WB, STAGE = 32 * (TA + TB);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wa = wave / WB, wb = wave % WB;
  const int s = lane & 15, g = lane >> 4;
  __bf16 *buf = (__bf16 *)lds;
  bf16x8 reg[NU];
  auto load = [&](int64_t row) {
#pragma unroll
    for (int k = 0; k < NU; ++k) {
      const int u = tid + k * DW_THREADS;
      reg[k] = bf16x8_zero();
      if (u < 32 * UA) {
        const int64_t r = row + u / UA;
        const int c = a0 + (u % UA) * 8;
        if (r < r1 && c < d.ka) reg[k] = *(const bf16x8 *)(d.A + r * d.lda + c);
      } else if (u < UNITS) {
        const int64_t r = row + (u - 32 * UA) / UB;
        const int c = ((u - 32 * UA) % UB) * 8;
        if (r < r1 && c < d.nb) reg[k] = *(const bf16x8 *)(d.B + r * d.ldb + c);
      }
    }
  };
  auto store = [&](__bf16 *b) {
#pragma unroll
    for (int k = 0; k < NU; ++k) {
      const int u = tid + k * DW_THREADS;
      if (u < 32 * UA) {
        const int r = u / UA, c = u % UA;
        *(bf16x8 *)(b + r * TA + ((c ^ dw_swizzle(r, UA)) << 3)) = reg[k];
      } else if (u < UNITS) {
        const int r = (u - 32 * UA) / UB, c = (u - 32 * UA) % UB;
        *(bf16x8 *)(b + 32 * TA + r * TB + ((c ^ dw_swizzle(r, UB)) << 3)) = reg[k];
      }
    }
  };
  // fragment of 16 columns from c0 of a staged operand of T columns
  auto frag = [&](const __bf16 *b, int T, int c0) {
    union { bf16x8 v; s16x4 h[2]; } f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = 8 * g + 4 * h + (s >> 2);
      const int unit = (c0 >> 3) + ((s & 3) >> 1);
      const __bf16 *p = b + row * T + ((unit ^ dw_swizzle(row, T / 8)) << 3) + (s & 1) * 4;
      f.h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p);
    }
    return f.v;
  };
  floatx4 acc[FA][FB];
  rows_zero<FA, FB>(acc);
  load(r0);
  store(buf);
  if (r0 + 32 < r1) load(r0 + 32);
  __syncthreads();
  int cur = 0;
  for (int64_t r = r0; r < r1; r += 32) {
    const __bf16 *b = buf + cur * STAGE;
    bf16x8 af[FA], bf[FB];
#pragma unroll
    for (int i = 0; i < FA; ++i) af[i] = frag(b, TA, (wa * FA + i) * 16);
#pragma unroll
    for (int j = 0; j < FB; ++j) bf[j] = frag(b + 32 * TA, TB, (wb * FB + j) * 16);
    // the other buffer was last read before the barrier that ended the step before
    if (r + 32 < r1) store(buf + (cur ^ 1) * STAGE);
    if (r + 64 < r1) load(r + 64);
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
      for (int j = 0; j < FB; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
    __syncthreads();
    cur ^= 1;
  }
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j) {
      const int n = (wb * FB + j) * 16 + s;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = a0 + (wa * FA + i) * 16 + g * 4 + r;
        if (k < d.ka && n < d.nb) part[(int64_t)k * d.nb + n] = acc[i][j][r];
      }
    }
}

template <int H>
__global__ void __launch_bounds__(DW_THREADS) mlp_weight_grad(DwArgs a) {
  __shared__ __align__(16) unsigned char lds[2 * 32 * (128 + H) * sizeof(__bf16)];
  static_assert(128 + H >= H + 32, "the thin tiles fit the same stages");
  constexpr int TILES = H / 128;  // tiles of an inner layer: 128 of its rows, all columns
  const int inner = (a.n_layers - 2) * TILES;
  const int b = blockIdx.x;
  const int l = b < inner ? 1 + b / TILES : (b == inner ? 0 : a.n_layers - 1);
  const DwLayer &d = a.layer[l];
  if ((int)blockIdx.y >= d.slices) return;
  const int64_t r0 = (int64_t)blockIdx.y * d.rows;
  const int64_t r1 = min(a.M, r0 + d.rows);
  float *part = d.part + (int64_t)blockIdx.y * d.ka * d.nb;
  if (b < inner) dw_tile<128, H, 2, 4>(d, (b % TILES) * 128, r0, r1, part, lds);
  else if (b == inner) dw_tile<K0, H, 1, 8>(d, 0, r0, r1, part, lds);
  else dw_tile<H, NOUT, 8, 1>(d, 0, r0, r1, part, lds);
}

// dW = sum of the slices in order; db = sum of the workgroups' column sums (blocks from
// dw_blocks on: 16 columns each, 16 chains of rows, then a tree)
__global__ void __launch_bounds__(256) mlp_grad_sums(DwArgs a, float *__restrict__ dW, int dw_blocks,
                                                     const float *__restrict__ dbp, int n_wg, int pitch, int n_db,
                                                     float *__restrict__ db) {
  if ((int)blockIdx.x < dw_blocks) {
    const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (e >= a.n_elems) return;
    int l = 0;
    while (l + 1 < a.n_layers && e >= a.layer[l + 1].off) ++l;
    const DwLayer &d = a.layer[l];
    const int S = d.slices;
    const int64_t n = (int64_t)d.ka * d.nb;
    const float *part = d.part + (e - d.off);
    floatx4 s = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
    for (int z = 0; z < S; ++z) {
      const floatx4 v = *(const floatx4 *)(part + z * n);
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] += v[r];
    }
    *(floatx4 *)(dW + e) = s;
    return;
  }
  __shared__ float t[16][17];
  const int col = ((int)blockIdx.x - dw_blocks) * 16 + (threadIdx.x & 15), q = threadIdx.x >> 4;
  float s = 0.0f;
  if (col < n_db)
    for (int k = q; k < n_wg; k += 16) s += dbp[(int64_t)k * pitch + col];
  t[q][threadIdx.x & 15] = s;
  __syncthreads();
  if (q == 0 && col < n_db) {
    float v = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; ++k) v += t[k][threadIdx.x];
    db[col] = v;
  }
}

struct Sizes {
  int64_t n_elems, part_elems, slices, wgs, db_pitch;  // slices: the most of any layer
  size_t g_bytes, gout_bytes, part_bytes, db_bytes;
  size_t total() const { return g_bytes + gout_bytes + part_bytes + db_bytes; }
};

// sizes of a backward pass; layer (optional): every layer's operand sizes and slices
Sizes train_sizes(int64_t M, int L, int k_in, int H, int np, DwLayer *layer = nullptr) {
  Sizes z{};
  for (int l = 0; l < L; ++l) {
    DwLayer d{};
    d.lda = d.ka = l == 0 ? k_in : H;
    d.ldb = l == L - 1 ? NOUT : H;
    d.nb = l == L - 1 ? np : H;
    gh::splitk_plan(d.ka, d.nb, (int)M, GH_EPI_STORE, d.slices, d.rows);
    d.off = z.n_elems;
    z.n_elems += (int64_t)d.ka * d.nb;
    z.part_elems += (int64_t)d.ka * d.nb * d.slices;
    z.slices = std::max<int64_t>(z.slices, d.slices);
    if (layer) layer[l] = d;
  }
  const int tile = 16 * row_tiles(M);
  z.wgs = (M + tile - 1) / tile;
  z.db_pitch = (int64_t)(L - 1) * H + NOUT;
  z.g_bytes = (size_t)(L - 1) * M * H * 2;
  z.gout_bytes = (size_t)M * NOUT * 2;
  z.part_bytes = (size_t)z.part_elems * 4;
  z.db_bytes = (size_t)z.wgs * z.db_pitch * 4;
  return z;
}

// n_out up to 16; parameter widths k_in and np are multiples of 8 (the tensors' padding)
bool sizes_ok(int64_t M, int L, int k_in, int H, int n_out, int np) {
  return M >= 1 && M <= GH_MLP_TRAIN_MAX_ROWS && L >= 2 && L <= MAXL && k_in >= 8 && k_in <= K0 && k_in % 8 == 0 &&
         (H == 128 || H == 256) && np >= 8 && np <= NOUT && np % 8 == 0 && n_out >= 1 && n_out <= np;
}

template <int H, int RT>
int launch_backward(const float *G, int64_t ldg, int64_t M, const BackArgs &a, hipStream_t st) {
  const dim3 grid((unsigned)((M + 16 * RT - 1) / (16 * RT)));
  constexpr size_t lds = rows_lds_bytes<H, RT>();
  const void *fn = (const void *)&mlp_rows_backward<H, RT>;
  if (lds + 1024 > 64 * 1024 &&
      hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return GH_EHIP;
  hipLaunchKernelGGL((mlp_rows_backward<H, RT>), grid, dim3(ROW_THREADS), lds, st, G, ldg, M, a);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}

bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

extern "C" int gh_mlp_train_forward_bf16(const void *X, int64_t M, int32_t n_layers, int32_t k_in, int32_t hidden,
                                         int32_t n_out, const void *const *wt, const float *const *bias,
                                         void *const *Y, float *Z, int64_t ldz, void *stream) {
  if (!X || !wt || !bias || !Y || !Z || ldz < n_out || !sizes_ok(M, n_layers, k_in, hidden, n_out, NOUT))
    return GH_EINVAL;
  MlpArgs a{};
  MlpKeep keep{};
  a.n_layers = n_layers;
  a.k_in = k_in;
  a.n_out = n_out;
  a.x_vec = 1;
  if (!aligned16(X)) return GH_EINVAL;
  for (int l = 0; l < n_layers; ++l) {
    if (!wt[l] || !bias[l] || !aligned16(wt[l]) || (l < n_layers - 1 && (!Y[l] || !aligned16(Y[l]) || !aligned16(bias[l]))))
      return GH_EINVAL;
    a.wt[l] = (const __bf16 *)wt[l];
    a.bias[l] = bias[l];
    if (l < n_layers - 1) keep.y[l] = (__bf16 *)Y[l];
  }
  const __bf16 *x = (const __bf16 *)X;
  hipStream_t st = (hipStream_t)stream;
  const int rt = row_tiles(M);
#define GH_ROWS(H)                                                                  \
  (rt == 1 ? launch_rows_forward<H, 1, true>(x, k_in, M, a, keep, Z, ldz, st)       \
           : (rt == 2 ? launch_rows_forward<H, 2, true>(x, k_in, M, a, keep, Z, ldz, st) \
                      : launch_rows_forward<H, 4, true>(x, k_in, M, a, keep, Z, ldz, st)))
  return hidden == 256 ? GH_ROWS(256) : GH_ROWS(128);
#undef GH_ROWS
}

extern "C" int gh_mlp_train_workspace(int64_t M, int32_t n_layers, int32_t k_in, int32_t hidden, int32_t np,
                                      int64_t *bytes) {
  if (!bytes || !sizes_ok(M, n_layers, k_in, hidden, np, np)) return GH_EINVAL;
  *bytes = (int64_t)train_sizes(M, n_layers, k_in, hidden, np).total();
  return GH_OK;
}

extern "C" int gh_mlp_train_backward_bf16(const void *X, int64_t M, int32_t n_layers, int32_t k_in, int32_t hidden,
                                          int32_t n_out, int32_t np, const void *const *w, const void *const *Y,
                                          const float *G, int64_t ldg, float *dW, float *db, float *const *G32, void *ws,
                                          int64_t ws_bytes, void *stream) {
  if (!X || !w || !Y || !G || !dW || !db || !ws || ldg < n_out || !sizes_ok(M, n_layers, k_in, hidden, n_out, np))
    return GH_EINVAL;
  const int L = n_layers;
  DwArgs d{};
  const Sizes z = train_sizes(M, L, k_in, hidden, np, d.layer);
  if (ws_bytes < (int64_t)z.total() || !aligned16(ws) || !aligned16(X) || !aligned16(dW)) return GH_EINVAL;
  for (int l = 0; l < L; ++l)
    if ((l > 0 && (!w[l] || !aligned16(w[l]))) ||
        (l < L - 1 && (!Y[l] || !aligned16(Y[l]) || (G32 && (!G32[l] || !aligned16(G32[l]))))))
      return GH_EINVAL;
  unsigned char *p = (unsigned char *)ws;  // every part is a multiple of 16 bytes
  BackArgs a{};
  a.n_layers = L;
  a.n_out = n_out;
  a.np = np;
  for (int l = 0; l < L - 1; ++l) {
    a.g[l] = (__bf16 *)(p + (size_t)l * M * hidden * 2);
    a.y[l] = (const __bf16 *)Y[l];
    if (G32) a.g32[l] = G32[l];
  }
  for (int l = 1; l < L; ++l) a.w[l] = (const __bf16 *)w[l];
  p += z.g_bytes;
  a.g_out = (__bf16 *)p;
  p += z.gout_bytes;
  float *part = (float *)p;
  p += z.part_bytes;
  a.db = (float *)p;
  hipStream_t st = (hipStream_t)stream;
  const int rt = row_tiles(M);
#define GH_ROWS(H)                                           \
  (rt == 1 ? launch_backward<H, 1>(G, ldg, M, a, st)         \
           : (rt == 2 ? launch_backward<H, 2>(G, ldg, M, a, st) : launch_backward<H, 4>(G, ldg, M, a, st)))
  const int rc = hidden == 256 ? GH_ROWS(256) : GH_ROWS(128);
#undef GH_ROWS
  if (rc != GH_OK) return rc;
  d.n_layers = L;
  d.M = M;
  d.n_elems = z.n_elems;
  for (int l = 0; l < L; ++l) {
    d.layer[l].A = l == 0 ? (const __bf16 *)X : a.y[l - 1];
    d.layer[l].B = l == L - 1 ? a.g_out : a.g[l];
    d.layer[l].part = part;
    part += (int64_t)d.layer[l].ka * d.layer[l].nb * d.layer[l].slices;
  }
  const dim3 grid((unsigned)((L - 2) * (hidden / 128) + 2), (unsigned)z.slices);
  if (hidden == 256) hipLaunchKernelGGL(mlp_weight_grad<256>, grid, dim3(DW_THREADS), 0, st, d);
  else hipLaunchKernelGGL(mlp_weight_grad<128>, grid, dim3(DW_THREADS), 0, st, d);
  if (hipGetLastError() != hipSuccess) return GH_EHIP;
  const int n_db = (L - 1) * hidden + np;
  const int dw_blocks = (int)((z.n_elems / 4 + 255) / 256);
  hipLaunchKernelGGL(mlp_grad_sums, dim3(dw_blocks + (n_db + 15) / 16), dim3(256), 0, st, d, dW, dw_blocks, a.db,
                     (int)z.wgs, (int)z.db_pitch, n_db, db);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}
