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
// register-held weights as the forward kernel (the rows of W_l [K][N] are the outputs of this
// product). The bias gradients are column sums of the FP32 gradients before
// their rounding to bf16: each workgroup writes the sums of its rows.
struct BackArgs {
  const __bf16 *w[MAXL];  // layer l >= 1: W_l [K_l][N_l] in fragment order (N of the last layer: 32)
  const __bf16 *y[MAXL];  // kept activations (MlpKeep order)
  __bf16 *g[MAXL];        // out: G_l for l <= L-2, in the same order
  __bf16 *g_out;          // out: bf16(G_{L-1}), 32 columns, in the same order
  float *g32[MAXL];       // out, optional: the FP32 gradients of the hidden layers, M x H
  float *db;              // out: [workgroup][(L-1) H + 16] partial sums (layer 0 first)
  int n_layers, n_out;
};

template <int H, int RT>
__global__ void __launch_bounds__(ROW_THREADS) mlp_rows_backward(const float *__restrict__ G, int64_t ldg, int64_t M,
                                                                 BackArgs a) {
  constexpr int NK = H / 32, CT = H / 128, ROWS = 16 * RT;
  extern __shared__ __align__(16) unsigned char mlp_lds[];
  __shared__ float s_last[ROW_THREADS / 64][NOUT];
  __bf16 *in = (__bf16 *)mlp_lds, *out = in + ROWS * H;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, g = lane >> 4;
  const int n0 = wave * 16 * CT;
  const int64_t row0 = (int64_t)blockIdx.x * ROWS;
  const int L = a.n_layers;
  float *db = a.db + (int64_t)blockIdx.x * ((L - 1) * H + NOUT);
  bf16x8 w0[CT], w[NK][CT];
#pragma unroll
  for (int j = 0; j < CT; ++j) w0[j] = *(const bf16x8 *)(a.w[L - 1] + ((wave * CT + j) * 64 + lane) * 8);
  // output gradient tile: bf16, padded to 32 columns
  for (int u = tid; u < ROWS * 4; u += ROW_THREADS) {
    const int r = u >> 2, q = (u & 3) * 8;
    const int64_t gr = row0 + r;
    bf16x8 v = bf16x8_zero();
    if (gr < M) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (q + j < a.n_out) v[j] = (__bf16)G[gr * ldg + q + j];
    }
    *(bf16x8 *)(in + (((r >> 4) * NK) * 64 + (u & 3) * 16 + (r & 15)) * 8) = v;
    if (gr < padded_rows(M)) *(bf16x8 *)(a.g_out + row0 * K0 + ((r >> 4) * 64 + (u & 3) * 16 + (r & 15)) * 8) = v;
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
  auto tiles = [&](int l) { return a.w[max(l, 1)] + wave * CT * NK * 512 + lane * 8; };
  auto fetch_y = [&](int l) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        const int64_t row = row0 + i * 16 + fr;
#pragma unroll
        for (int r = 0; r < 4; ++r) y[i][j][r] = (__bf16)0.0f;
        if (row < M) y[i][j] = *(const bf16x4 *)(a.y[l] + row0 * H + rows_at<NK>(i, fr, n0 + j * 16 + g * 4));
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
        // (rows from M on are exact zeros: their output gradients are)
        const int64_t row = row0 + i * 16 + fr;
        if (row < padded_rows(M)) *(bf16x4 *)(a.g[l] + row0 * H + rows_at<NK>(i, fr, c)) = v;
        if (a.g32[l] && row < M) *(floatx4 *)(a.g32[l] + row * H + c) = z;
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
  fetch_y(L - 2);
  if (L > 2) rows_weights<CT, NK>(w, tiles(L - 2), NK * 512);
  __syncthreads();
  if (tid < NOUT) {
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < ROW_THREADS / 64; ++k) s += s_last[k][tid];
    db[(L - 1) * H + tid] = s;
  }
  rows_zero<RT, CT>(acc);
  rows_mma0<RT, CT, NK>(acc, w0, in, lane);
  finish(L - 2);
  for (int l = L - 2; l >= 1; --l) {  // G_{l-1} from G_l
    fetch_y(l - 1);
    rows_zero<RT, CT>(acc);
    rows_mma<RT, CT, NK>(acc, w, in, lane, tiles(l - 1), NK * 512);
    finish(l - 1);
  }
}

// ------------------------------------------------------------------ weight gradients
// dW_l = X_l^T G_l: reductions over the batch of two matrices in MlpKeep order (tiles of 16
// rows; the input and the output gradient padded to 32 columns, all to a multiple of 32 rows
// with zeros). All layers in one launch: blockIdx.x is an output tile of some layer, blockIdx.y
// a slice of the rows. The slices are those of gh_gemm_bf16 for the same product (its rule: 512
// rows from 2048 rows on, 32 slices and 256 workgroups for the four inner layers at 16384
// rows), so the sums have the same bits. A step of 32 rows (512 MFMA cycles) is shorter than the
// latency of its 24 KiB: the steps come through a ring of three LDS stages (two workgroups of
// 72 KiB per CU), two in flight, by direct global-to-LDS loads of 1 KiB blocks. The fragments (8 consecutive rows of one
// column) are read with the transposing LDS read (ds_read_b64_tr_b16: lane s of 16 names 4
// columns of row s / 4, lane i receives 4 rows of column i); the 16-byte units of odd column
// groups sit at row ^ 4, so that the 8 rows and 2 groups of a half wave fall into different
// banks.
struct DwLayer {
  const __bf16 *A, *B;  // X_l and G_l
  int na, nb32;         // 32-column blocks per row tile of A and B
  int ka, nb;           // valid columns of A and B: dW_l is ka x nb
  int rows, slices;     // rows of a slice, number of slices
  float *part;          // [slice][ka nb] partial sums
  int64_t off;          // offset of the layer's ka x nb block in the result
};
struct DwArgs {
  DwLayer layer[MAXL];
  int n_layers;
  int64_t M, n_elems;   // elements of the result
};

constexpr int DW_THREADS = 512, DW_STAGES = 3;

// 16 bytes per lane to LDS at p + 16 lane, p wave-uniform. In asm, so that the compiler does
// not put its own wait for every load in flight in front of each LDS read and barrier: the
// caller waits (vmcnt) and then meets a barrier before it reads. No vector register is
// written; m0 is set where it is used, as the compiler does for its own loads.
__device__ __forceinline__ void lds_load(const void *p, const void *src) {
  const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)p;
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(__builtin_amdgcn_readfirstlane(at)), "v"(src)
               : "memory");
}

// output tile [a0, a0 + TA) x [0, TB) over the waves WA x WB, FA x FB fragments each
template <int TA, int TB, int WA, int WB, int FA, int FB>
__device__ __forceinline__ void dw_tile(const DwLayer &d, int a0, int64_t r0, int64_t r1, float *part,
                                        unsigned char *lds) {
  constexpr int BA = TA / 32, BB = TB / 32, BLOCKS = 2 * (BA + BB), PER_WAVE = (BLOCKS + 7) / 8;
  constexpr int STAGE = BLOCKS * 512;  // elements
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wa = wave / WB, wb = wave % WB;
  const int s = lane & 15, g = lane >> 4;
  __bf16 *buf = (__bf16 *)lds;
  const int swz = ((lane >> 4) & 1) << 2;  // of the unit (column group lane / 16, row lane % 16)
  const int steps = (int)((r1 - r0 + 31) >> 5);
  // block b of a stage: row tile b / (BA + BB), then A's blocks, then B's; a wave without a
  // PER_WAVE-th block loads an earlier one again, so that every wave waits for the same count
  const __bf16 *src[PER_WAVE];
  int stride[PER_WAVE];  // per step
#pragma unroll
  for (int k = 0; k < PER_WAVE; ++k) {
    const int b = (wave + 8 * k) % BLOCKS;
    const int64_t tile = (r0 >> 4) + b / (BA + BB);
    const int q = b % (BA + BB);
    src[k] = (q < BA ? d.A + (tile * d.na + (a0 >> 5) + q) * 512 : d.B + (tile * d.nb32 + (q - BA)) * 512) +
             (lane ^ swz) * 8;
    stride[k] = (q < BA ? d.na : d.nb32) * 1024;
  }
  auto load = [&](int t) {
    const __bf16 *stage = buf + (t % DW_STAGES) * STAGE;
#pragma unroll
    for (int k = 0; k < PER_WAVE; ++k)
      lds_load(stage + ((wave + 8 * k) % BLOCKS) * 512, src[k] + (int64_t)t * stride[k]);
  };
  // fragment of 16 columns from c0 of a staged operand whose first block is b0
  auto frag = [&](const __bf16 *stage, int b0, int c0) {
    union { bf16x8 v; s16x4 h[2]; } f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = 8 * (g & 1) + 4 * h + (s >> 2);  // in row tile g / 2
      const int c = c0 + 4 * (s & 3), kg = (c >> 3) & 3;
      const __bf16 *p = stage + ((g >> 1) * (BA + BB) + b0 + (c >> 5)) * 512 +
                        (kg * 16 + (row ^ ((kg & 1) << 2))) * 8 + (c & 4);
      f.h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p);
    }
    return f.v;
  };
  floatx4 acc[FA][FB];
  rows_zero<FA, FB>(acc);
#pragma unroll
  for (int t = 0; t < DW_STAGES - 1; ++t)
    if (t < steps) load(t);
  for (int t = 0; t < steps; ++t) {
    // this wave's blocks of step t have arrived (loads return in order; the next step's in
    // flight) and its LDS reads of step t - 1 are done; after the barrier that holds for
    // every wave, and the next load may refill the stage of step t - 1
    if (t + 1 < steps) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(PER_WAVE) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + DW_STAGES - 1 < steps) load(t + DW_STAGES - 1);
    const __bf16 *stage = buf + (t % DW_STAGES) * STAGE;
    bf16x8 af[FA], bf[FB];
#pragma unroll
    for (int i = 0; i < FA; ++i) af[i] = frag(stage, 0, (wa * FA + i) * 16);
#pragma unroll
    for (int j = 0; j < FB; ++j) bf[j] = frag(stage, BA, (wb * FB + j) * 16);
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
      for (int j = 0; j < FB; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
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
  extern __shared__ __align__(16) unsigned char lds[];  // DW_STAGES stages of 32 rows x (128 + H) columns
  constexpr int TILES = H / 128;  // tiles of an inner layer: 128 of its rows, all columns
  const int inner = (a.n_layers - 2) * TILES;
  const int b = blockIdx.x;
  const int l = b < inner ? 1 + b / TILES : (b == inner ? 0 : a.n_layers - 1);
  const DwLayer &d = a.layer[l];
  if ((int)blockIdx.y >= d.slices) return;
  const int64_t r0 = (int64_t)blockIdx.y * d.rows;
  const int64_t r1 = min(a.M, r0 + d.rows);
  float *part = d.part + (int64_t)blockIdx.y * d.ka * d.nb;
  if (b < inner) dw_tile<128, H, 2, 4, 4, H / 64>(d, (b % TILES) * 128, r0, r1, part, lds);
  else if (b == inner) dw_tile<K0, H, 1, 8, 2, H / 128>(d, 0, r0, r1, part, lds);
  else dw_tile<H, K0, 8, 1, H / 128, 1>(d, 0, r0, r1, part, lds);
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
    d.ka = l == 0 ? k_in : H;
    d.na = l == 0 ? 1 : H / 32;
    d.nb = l == L - 1 ? np : H;
    d.nb32 = l == L - 1 ? 1 : H / 32;
    gh::splitk_plan(d.ka, d.nb, (int)M, GH_EPI_STORE, d.slices, d.rows);
    d.off = z.n_elems;
    z.n_elems += (int64_t)d.ka * d.nb;
    z.part_elems += (int64_t)d.ka * d.nb * d.slices;
    z.slices = std::max<int64_t>(z.slices, d.slices);
    if (layer) layer[l] = d;
  }
  z.wgs = row_grid(M, row_tiles(M));
  z.db_pitch = (int64_t)(L - 1) * H + NOUT;
  z.g_bytes = (size_t)(L - 1) * padded_rows(M) * H * 2;
  z.gout_bytes = (size_t)padded_rows(M) * K0 * 2;
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
  const dim3 grid((unsigned)row_grid(M, RT));
  constexpr size_t lds = rows_lds_bytes<H, RT>();
  const void *fn = (const void *)&mlp_rows_backward<H, RT>;
  if (lds + 1024 > 64 * 1024 &&
      hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return GH_EHIP;
  hipLaunchKernelGGL((mlp_rows_backward<H, RT>), grid, dim3(ROW_THREADS), lds, st, G, ldg, M, a);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}

bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// ------------------------------------------------------------------ column sums
// Sums over the rows of several FP32 matrices, in one fixed order of additions: workgroup c of
// `ctas` and its thread row y of `by` add the rows s + S i, s = c by + y and S = by ctas, in
// four running sums (i mod 4), then those, then the thread rows by halves, then the workgroups
// (y, y + by, ... and the thread rows by halves again). This is the order in which PyTorch
// 2.10.0 sums the columns of a matrix of these widths, found by comparing bits over 1..70000 rows
// (tests/test_gpu_column_sums.py holds it; another version may sum in another order, this one does
// not change): fits divide by the size of nearly cancelled sums in their first steps, so another
// order gives other weights. PyTorch's calls, one a layer, took 125 us for 5 x 16384 x 256 and 32
// for 3 x 5003 x 128; these two launches 23 and 15, the first bound by reading 84 MB from behind
// the L2 (5.2 TB/s), the second by the one workgroup of its last layer.
struct ColSum {
  const float *g;
  int64_t ld;
  int n, n_pad;    // columns, and with the zero columns behind them
  int by, ctas;
  float *part;     // [ctas][n_pad]
  float *out;      // n_pad
};
struct ColSums {
  ColSum m[MAXL];
  int64_t M;
};
constexpr int COLSUM_THREADS = 128;

// thread rows and workgroups of a matrix of M x n rows
void column_plan(int64_t M, int n_pad, int &by, int &ctas) {
  by = COLSUM_THREADS / (n_pad / 4);
  if (M < 16 * by && M < 256) by = 1;
  const int64_t rows = (M + by - 1) / by, want = (rows + 15) / 16;
  ctas = rows < 256 ? 1 : (want <= 128 ? (int)want : (want <= 256 ? 128 : 256));
}

__device__ __forceinline__ float4 add4(float4 a, float4 b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

__global__ void __launch_bounds__(COLSUM_THREADS) column_part_kernel(ColSums C) {
  const ColSum m = C.m[blockIdx.y];
  if ((int)blockIdx.x >= m.ctas) return;
  __shared__ float4 s_v[COLSUM_THREADS];
  const int groups = m.n_pad / 4, t = threadIdx.x, col = (t % groups) * 4, y = t / groups;
  float4 a[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) a[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  auto rows = [&](auto load) {
    const int64_t S = (int64_t)m.by * m.ctas;
    int64_t r = (int64_t)blockIdx.x * m.by + y;
#pragma unroll 4
    for (; r + 3 * S < C.M; r += 4 * S) {
      float4 v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = load(m.g + (r + k * S) * m.ld + col);
#pragma unroll
      for (int k = 0; k < 4; ++k) a[k] = add4(a[k], v[k]);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (r + k * S < C.M) a[k] = add4(a[k], load(m.g + (r + k * S) * m.ld + col));
  };
  if (y < m.by && col < m.n) {
    if ((m.ld & 3) == 0 && col + 4 <= m.n && ((uintptr_t)m.g & 15) == 0) {
      rows([](const float *p) { return *(const float4 *)p; });
    } else {
      const int left = m.n - col;
      rows([left](const float *p) {
        return make_float4(p[0], left > 1 ? p[1] : 0.0f, left > 2 ? p[2] : 0.0f, left > 3 ? p[3] : 0.0f);
      });
    }
  }
  float4 v = add4(add4(add4(a[0], a[1]), a[2]), a[3]);
  for (int o = m.by / 2; o > 0; o >>= 1) {
    s_v[t] = v;
    __syncthreads();
    if (y < o) v = add4(v, s_v[t + o * groups]);
    __syncthreads();
  }
  if (y == 0) *(float4 *)((m.ctas > 1 ? m.part + (int64_t)blockIdx.x * m.n_pad : m.out) + col) = v;
}

__global__ void __launch_bounds__(COLSUM_THREADS) column_total_kernel(ColSums C) {
  const ColSum m = C.m[blockIdx.y];
  const int cols = COLSUM_THREADS / m.by, t = threadIdx.x, col = (int)blockIdx.x * cols + t % cols, y = t / cols;
  if (m.ctas == 1 || (int)blockIdx.x * cols >= m.n_pad) return;
  __shared__ float s_v[COLSUM_THREADS];
  float v = 0.0f;
  if (col < m.n_pad) {
#pragma unroll 8
    for (int c = y; c < m.ctas; c += m.by) v += m.part[(int64_t)c * m.n_pad + col];
  }
  for (int o = m.by / 2; o > 0; o >>= 1) {
    s_v[t] = v;
    __syncthreads();
    if (y < o) v += s_v[t + o * cols];
    __syncthreads();
  }
  if (y == 0 && col < m.n_pad) m.out[col] = v;
}

}  // namespace

extern "C" int gh_mlp_train_forward_bf16(const void *X, int64_t M, int32_t n_layers, int32_t k_in, int32_t hidden,
                                         int32_t n_out, const void *const *wt, const float *const *bias, void *Xt,
                                         void *const *Y, float *Z, int64_t ldz, void *stream) {
  if (!X || !wt || !bias || !Xt || !aligned16(Xt) || !Y || !Z || ldz < n_out || !sizes_ok(M, n_layers, k_in, hidden, n_out, NOUT))
    return GH_EINVAL;
  MlpArgs a{};
  MlpKeep keep{};
  a.n_layers = n_layers;
  a.k_in = k_in;
  a.n_out = n_out;
  a.x_vec = 1;
  keep.x = (__bf16 *)Xt;
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
  (rt == 1 ? launch_rows_forward<H, 1, 8, ROWS_KEEP>(x, k_in, M, a, keep, {}, Z, ldz, st)       \
           : (rt == 2 ? launch_rows_forward<H, 2, 8, ROWS_KEEP>(x, k_in, M, a, keep, {}, Z, ldz, st) \
                      : launch_rows_forward<H, 4, 8, ROWS_KEEP>(x, k_in, M, a, keep, {}, Z, ldz, st)))
  return hidden == 256 ? GH_ROWS(256) : GH_ROWS(128);
#undef GH_ROWS
}

extern "C" int gh_mlp_train_workspace(int64_t M, int32_t n_layers, int32_t k_in, int32_t hidden, int32_t np,
                                      int64_t *bytes) {
  if (!bytes || !sizes_ok(M, n_layers, k_in, hidden, np, np)) return GH_EINVAL;
  *bytes = (int64_t)train_sizes(M, n_layers, k_in, hidden, np).total();
  return GH_OK;
}

extern "C" int gh_mlp_train_backward_bf16(const void *Xt, int64_t M, int32_t n_layers, int32_t k_in, int32_t hidden,
                                          int32_t n_out, int32_t np, const void *const *w, const void *const *Y,
                                          const float *G, int64_t ldg, float *dW, float *db, float *const *G32, void *ws,
                                          int64_t ws_bytes, void *stream) {
  if (!Xt || !w || !Y || !G || !dW || !db || !ws || ldg < n_out || !sizes_ok(M, n_layers, k_in, hidden, n_out, np))
    return GH_EINVAL;
  const int L = n_layers;
  DwArgs d{};
  const Sizes z = train_sizes(M, L, k_in, hidden, np, d.layer);
  if (ws_bytes < (int64_t)z.total() || !aligned16(ws) || !aligned16(Xt) || !aligned16(dW)) return GH_EINVAL;
  for (int l = 0; l < L; ++l)
    if ((l > 0 && (!w[l] || !aligned16(w[l]))) ||
        (l < L - 1 && (!Y[l] || !aligned16(Y[l]) || (G32 && (!G32[l] || !aligned16(G32[l]))))))
      return GH_EINVAL;
  unsigned char *p = (unsigned char *)ws;  // every part is a multiple of 16 bytes
  BackArgs a{};
  a.n_layers = L;
  a.n_out = n_out;
  for (int l = 0; l < L - 1; ++l) {
    a.g[l] = (__bf16 *)(p + (size_t)l * padded_rows(M) * hidden * 2);
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
    d.layer[l].A = l == 0 ? (const __bf16 *)Xt : a.y[l - 1];
    d.layer[l].B = l == L - 1 ? a.g_out : a.g[l];
    d.layer[l].part = part;
    part += (int64_t)d.layer[l].ka * d.layer[l].nb * d.layer[l].slices;
  }
  const dim3 grid((unsigned)((L - 2) * (hidden / 128) + 2), (unsigned)z.slices);
  const size_t lds = (size_t)DW_STAGES * 32 * (128 + hidden) * sizeof(__bf16);
  if (hidden == 256) {
    if (hipFuncSetAttribute((const void *)&mlp_weight_grad<256>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds) != hipSuccess)
      return GH_EHIP;
    hipLaunchKernelGGL(mlp_weight_grad<256>, grid, dim3(DW_THREADS), lds, st, d);
  } else {
    hipLaunchKernelGGL(mlp_weight_grad<128>, grid, dim3(DW_THREADS), lds, st, d);
  }
  if (hipGetLastError() != hipSuccess) return GH_EHIP;
  const int n_db = (L - 1) * hidden + np;
  const int dw_blocks = (int)((z.n_elems / 4 + 255) / 256);
  hipLaunchKernelGGL(mlp_grad_sums, dim3(dw_blocks + (n_db + 15) / 16), dim3(256), 0, st, d, dW, dw_blocks, a.db,
                     (int)z.wgs, (int)z.db_pitch, n_db, db);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}

extern "C" int gh_column_sums(const float *const *G, const int64_t *ld, const int32_t *n, const int32_t *n_pad,
                              int32_t count, int64_t M, float *const *out, float *work, int64_t work_floats,
                              void *stream) {
  if (!G || !ld || !n || !n_pad || !out || !work || count <= 0 || count > MAXL || M <= 0 ||
      M > GH_COLUMN_SUMS_MAX_ROWS || !aligned16(work))
    return GH_EINVAL;
  ColSums c{};
  c.M = M;
  int ctas = 1, blocks = 1;
  int64_t used = 0;
  for (int k = 0; k < count; ++k) {
    const int w = n_pad[k];
    if (!G[k] || !out[k] || !aligned16(out[k]) || n[k] <= 0 || n[k] > w || ld[k] < n[k] || w < 8 || w > 256 ||
        (w & (w - 1)) != 0)
      return GH_EINVAL;
    ColSum &m = c.m[k];
    m.g = G[k]; m.ld = ld[k]; m.n = n[k]; m.n_pad = w; m.out = out[k];
    column_plan(M, w, m.by, m.ctas);
    m.part = work + used;
    if (m.ctas > 1) {
      used += (int64_t)m.ctas * w;
      blocks = std::max(blocks, (w * m.by + COLSUM_THREADS - 1) / COLSUM_THREADS);
    }
    ctas = std::max(ctas, m.ctas);
  }
  if (work_floats < used) return GH_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(column_part_kernel, dim3(ctas, count), dim3(COLSUM_THREADS), 0, st, c);
  if (ctas > 1) hipLaunchKernelGGL(column_total_kernel, dim3(blocks, count), dim3(COLSUM_THREADS), 0, st, c);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}
