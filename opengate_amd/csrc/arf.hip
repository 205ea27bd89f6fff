// SPECT detection for the learned detector response (ARF) and for its plain-transport
// counterpart.
//
// gh_spect_pairs: photons that left the phantom (exit point p, direction d, vacuum
// outside) are projected onto every detector head of the gantry. Head k sits at angle
// a_k around the z axis through `center`, with outward normal n_k = (cos a_k, sin a_k, 0)
// and tangential axis e_k = (-sin a_k, cos a_k, 0); its collimator face is the plane
// (x - center).n_k = radius. A photon reaches head k when c = d.n_k > cos(theta_max)
// (larger incidence angles are absorbed by the collimator); it crosses the face at
// h = p + t d, t = (radius - (p - center).n_k)/c, and is binned at the crossing of the
// plane crystal_depth further (GateARFActor: distance_to_crystal). In the head frame
// x' = axial (z), y' = tangential, z' = -n_k (towards the source) the direction is
// d' = (d_z, d.e_k, -c); theta = acos(c), phi = atan2(d'_y, d'_x)
// (GateARFTrainingDatasetActor.cpp:99-107 with the plane normal as third axis).
// Every (photon, head) pair is written to a slot that its workgroup reserved: the NN input
// row (bf16: E, theta, phi scaled by norm[]), the pixel index (head*ny + iy)*nx + ix,
// the weight, and optionally the photon in the frame of a detector model whose hexagonal
// hole lattice (pitch, first lattice vector along x') has a lattice point at
// patch_origin: the entry point is reduced to the lattice cell, so a finite model patch
// stands for the whole periodic collimator.
//
// gh_energy_windows: deposited energy per event -> energy window (0 = none) after a
// Gaussian blur whose width follows one of the digitizer laws (fixed sigma, inverse-square
// root FWHM = resolution sqrt(reference E), linear FWHM/E), noise from Philox4x32-10
// (key = seed, counter = (event lo, event hi, "BLUR", 0)).
//
// gh_arf_accumulate / gh_counts_accumulate: add the window probabilities of the network
// (softmax of its n_win+1 logits, class 0 = not detected) or the simulated window of
// each pair into projection images [head][window][ny][nx] (FP64 atomics), optionally
// the squared contributions too.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "../../include/gatehip.h"
#include "gh_device.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

namespace {

using namespace gh;

constexpr uint32_t BLUR_TAG = 0x424C5552u;  // "BLUR"
constexpr int MAX_WIN = 8;

struct PairOut {
  __bf16 *x16;
  int32_t *pix;
  float *wgt;
  float *det[8];
  float *tp;
  unsigned long long *count;
  int64_t capacity;
};

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }
__device__ __forceinline__ uint32_t mbcnt(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Pairs found by a workgroup wait in LDS until PAIR_CAP could overflow, and then take their slots
// with one atomic: all slots come from one counter, which serves an atomic every 12 ns wherever it
// comes from. (One atomic for each wave and 64 tested heads was that bound: 10^6 photons on 128 heads,
// 500 us; so 46.) The waiting pairs hold what the geometry needs anyway; angles and
// rows are computed when they are written, by full waves.
constexpr int PAIR_CAP = 768;

template <bool DET>
__global__ void __launch_bounds__(256) spect_pairs_kernel(const float *__restrict__ x, const float *__restrict__ y,
                                                          const float *__restrict__ z, const float *__restrict__ u,
                                                          const float *__restrict__ v, const float *__restrict__ w,
                                                          const float *__restrict__ E, const float *__restrict__ wt,
                                                          int64_t n, gh_spect_desc D, const float *__restrict__ cs,
                                                          PairOut o) {
  enum { PX, PY, PZ, DU, DV, DW, EN, WT, CAND_FIELDS };
  enum { C, DY, QW, QE, QWT, HU, HZ, PAIR_FIELDS };
  __shared__ float s_cand[CAND_FIELDS][256];
  __shared__ int s_k0[256];
  __shared__ float s_pair[DET ? PAIR_FIELDS : HU][PAIR_CAP];
  __shared__ int s_pix[PAIR_CAP];
  __shared__ int s_n[2][2][4];  // of candidates and of pairs, by wave; two in turn: one barrier a round
  __shared__ unsigned long long s_slot;
  const int wave = (int)(threadIdx.x >> 6);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const float two_pi = 6.28318530717958647692f;
  const float dalpha = two_pi / (float)D.n_proj;
  const float sin_max = sqrtf(fmaxf(fmaf(-D.cos_theta_max, D.cos_theta_max, 1.0f), 0.0f));
  // candidate heads: |azimuth(d) - a_k| < theta_max, so k0 +- margin covers them; when
  // that window wraps onto itself every head is visited once instead
  int margin = (int)ceilf(asinf(fminf(sin_max, 1.0f)) / dalpha) + 2;
  const bool all_heads = 2 * margin + 1 >= D.n_proj;
  const int jlo = all_heads ? 0 : -margin, jhi = all_heads ? D.n_proj - 1 : margin;
  const float half_w = 0.5f * (float)D.nx * D.spacing[0], half_h = 0.5f * (float)D.ny * D.spacing[1];
  const float a2x = 0.5f * D.pitch, a2y = 0.86602540378443865f * D.pitch;
  int waiting = 0;  // the same in every thread, as every bound of the loops below

  // position of this lane's item among those of the workgroup; every thread gets their number
  auto place = [&](int (&counts)[4], bool mine, int &total) {
    const uint64_t m = __ballot(mine);
    if (lane_id() == 0) counts[wave] = __popcll(m);
    __syncthreads();
    int before = 0;
    total = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q < wave) before += counts[q];
      total += counts[q];
    }
    return before + (int)mbcnt(m);
  };

  auto write_out = [&]() {
    __syncthreads();
    if (threadIdx.x == 0) s_slot = atomicAdd(o.count, (unsigned long long)waiting);
    __syncthreads();
    for (int p = (int)threadIdx.x; p < waiting; p += 256) {
      const uint64_t slot = s_slot + (uint64_t)p;
      if ((int64_t)slot >= o.capacity) break;
      const float c = s_pair[C][p], dy = s_pair[DY][p], qw = s_pair[QW][p], qe = s_pair[QE][p];
      const float theta = acosf(fminf(c, 1.0f));
      const float phi = atan2f(dy, qw);
      if (o.x16) {
        bf16x8 row = {};
        row[0] = (__bf16)fmaf(qe, D.norm[0], D.norm[1]);
        row[1] = (__bf16)fmaf(theta, D.norm[2], D.norm[3]);
        row[2] = (__bf16)fmaf(phi, D.norm[4], D.norm[5]);
        __builtin_memcpy(o.x16 + slot * 8, &row, sizeof(row));
      }
      if (o.tp) { o.tp[2 * slot] = theta; o.tp[2 * slot + 1] = phi; }
      o.pix[slot] = s_pix[p];
      o.wgt[slot] = s_pair[QWT][p];
      if constexpr (DET) {
        // head frame: x' axial (hz), y' tangential (hu); reduce to the lattice cell
        float rx = s_pair[HZ][p], ry = s_pair[HU][p];
        if (D.pitch > 0.0f) {
          const float jj = floorf(ry / a2y);
          ry = fmaf(-jj, a2y, ry);
          rx = fmaf(-jj, a2x, rx);
          const float ii = floorf(rx / D.pitch);
          rx = fmaf(-ii, D.pitch, rx);
        }
        o.det[0][slot] = D.patch_origin[0] + rx;
        o.det[1][slot] = D.patch_origin[1] + ry;
        o.det[2][slot] = D.patch_origin[2];
        o.det[3][slot] = qw;
        o.det[4][slot] = dy;
        o.det[5][slot] = -c;
        o.det[6][slot] = qe;
        o.det[7][slot] = s_pair[QWT][p];
      }
    }
    __syncthreads();
    waiting = 0;
  };

  int turn = 0, round = 0;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < n; base += stride, turn ^= 1) {
    const int64_t i = base + threadIdx.x;
    float du = 0.f, dv = 0.f, dw = 1.f, ww = 0.f;
    bool cand = false;
    if (i < n) {
      du = u[i]; dv = v[i]; dw = w[i]; ww = wt[i];
      // only directions within theta_max of the transverse plane can reach a head
      cand = fabsf(dw) < sin_max && ww > 0.0f;
    }
    int n_cand;
    const int at = place(s_n[0][turn], cand, n_cand);
    if (cand) {
      int k0 = 0;
      if (!all_heads) {
        const float beta = atan2f(dv, du) - D.angle0;
        k0 = (int)floorf(beta / dalpha + 0.5f);
      }
      s_k0[at] = k0;
      s_cand[PX][at] = x[i] - D.center[0];
      s_cand[PY][at] = y[i] - D.center[1];
      s_cand[PZ][at] = z[i] - D.center[2];
      s_cand[DU][at] = du; s_cand[DV][at] = dv; s_cand[DW][at] = dw;
      s_cand[EN][at] = E[i];
      s_cand[WT][at] = ww;
    }
    __syncthreads();
    // the (candidate photon, head) items of the workgroup over its 256 threads
    const int width = jhi - jlo + 1;
    const int64_t n_items = (int64_t)n_cand * width;
    for (int64_t it0 = 0; it0 < n_items; it0 += 256, round ^= 1) {
      if (waiting > PAIR_CAP - 256) write_out();
      const int64_t item = it0 + (int64_t)threadIdx.x;
      bool hit = false;
      int32_t pixel = 0;
      int ci = 0;
      float c = 0.f, dy = 0.f, hu = 0.f, hz = 0.f;
      if (item < n_items) {
        ci = n_items <= INT32_MAX ? (int)((uint32_t)item / (uint32_t)width) : (int)(item / width);
        const int j = jlo + (int)(item - (int64_t)ci * width);
        const float px = s_cand[PX][ci], py = s_cand[PY][ci], pz = s_cand[PZ][ci];
        const float du = s_cand[DU][ci], dv = s_cand[DV][ci], dw = s_cand[DW][ci];
        const int k = ((s_k0[ci] + j) % D.n_proj + D.n_proj) % D.n_proj;
        const float ca = cs[2 * k], sa = cs[2 * k + 1];
        c = fmaf(du, ca, dv * sa);
        if (c > D.cos_theta_max) {
          const float s = fmaf(px, ca, py * sa);
          const float t = (D.radius - s) / c;
          if (t >= 0.0f) {
            dy = fmaf(-du, sa, dv * ca);  // d . e_k
            const float ex = fmaf(t, du, px), ey = fmaf(t, dv, py);
            hu = fmaf(-ex, sa, ey * ca);  // tangential coordinate on the face
            hz = fmaf(t, dw, pz);         // axial coordinate on the face
            const float f = D.crystal_depth / c;
            const float bu = fmaf(f, dy, hu), bz = fmaf(f, dw, hz);
            const float fx = (bu + half_w) / D.spacing[0], fy = (bz + half_h) / D.spacing[1];
            if (fx >= 0.0f && fy >= 0.0f && fx < (float)D.nx && fy < (float)D.ny) {
              const int ix = min((int)fx, D.nx - 1), iy = min((int)fy, D.ny - 1);
              pixel = (k * D.ny + iy) * D.nx + ix;
              hit = true;
            }
          }
        }
      }
      int found;
      const int p = waiting + place(s_n[1][round], hit, found);
      if (hit) {
        s_pix[p] = pixel;
        s_pair[C][p] = c;
        s_pair[DY][p] = dy;
        s_pair[QW][p] = s_cand[DW][ci];
        s_pair[QE][p] = s_cand[EN][ci];
        s_pair[QWT][p] = s_cand[WT][ci];
        if constexpr (DET) {
          s_pair[HU][p] = hu;
          s_pair[HZ][p] = hz;
        }
      }
      waiting += found;
    }
  }
  if (waiting) write_out();
}

struct Windows {
  float lo[MAX_WIN], hi[MAX_WIN];
  int n;
};

// standard deviation of the blurred energy of an event with energy e (MeV); FWHM laws are
// converted with 1 / (2 sqrt(2 ln 2))
__device__ __forceinline__ float blur_sigma(const gh_blur &B, float e) {
  constexpr float fwhm_to_sigma = 0.42466090014400953f;
  if (B.law == GH_BLUR_GAUSSIAN) return B.sigma;
  if (B.law == GH_BLUR_INVERSE_SQUARE) return (B.resolution * sqrtf(B.reference * e)) * fwhm_to_sigma;
  return ((B.slope * (e - B.reference) + B.resolution) * e) * fwhm_to_sigma;
}

__global__ void __launch_bounds__(256) energy_windows_kernel(const float *__restrict__ edep, int64_t n, uint32_t k0,
                                                             uint32_t k1, uint64_t first, gh_blur B, Windows W,
                                                             int32_t *__restrict__ cls) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float e = edep[i];
    int c = 0;
    if (e > 0.0f) {
      float eb = e;
      if (B.law != GH_BLUR_NONE) {
        const uint64_t id = first + (uint64_t)i;
        uint32_t x0 = (uint32_t)id, x1 = (uint32_t)(id >> 32), x2 = BLUR_TAG, x3 = 0u;
        philox10(x0, x1, x2, x3, k0, k1);
        const float u0 = (float)((x0 >> 8) | 1u) * 0x1p-24f, u1 = (float)((x1 >> 8) | 1u) * 0x1p-24f;
        float sn, csn;
        gsincos(6.28318530717958647692f * u1, sn, csn);
        const float g = sqrtf(-2.0f * glog(u0, c_logtab)) * csn;
        eb = fmaf(blur_sigma(B, e), g, e);
      }
      for (int k = 0; k < W.n; ++k)
        if (eb >= W.lo[k] && eb < W.hi[k]) { c = k + 1; break; }
    }
    cls[i] = c;
  }
}

__device__ __forceinline__ void add_f64(double *p, double v) {
  __builtin_amdgcn_global_atomic_fadd_f64((__attribute__((address_space(1))) double *)p, v);
}

// p[k] = weight x softmax(l)[k + 1], k < n_win <= N
template <int N>
__device__ __forceinline__ void softmax_row(const float *__restrict__ l, int n_win, float weight, float (&p)[N]) {
  float mx = l[0];
  for (int k = 1; k <= n_win; ++k) mx = fmaxf(mx, l[k]);
  float s = 0.0f;
  for (int k = 0; k <= n_win; ++k) s += __expf(l[k] - mx);
  const float inv = weight / s;
#pragma unroll
  for (int k = 0; k < N; ++k)
    if (k < n_win) p[k] = __expf(l[k + 1] - mx) * inv;
}

__global__ void __launch_bounds__(256) arf_accumulate_kernel(const float *__restrict__ logits, int64_t ldl, int64_t m,
                                                             const int32_t *__restrict__ pix,
                                                             const float *__restrict__ wgt, int n_win, int plane,
                                                             double *img, double *img2) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < m; r += stride) {
    float p[MAX_WIN];
    softmax_row(logits + r * ldl, n_win, wgt[r], p);
    const int32_t q = pix[r];
    const int32_t head = q / plane, rem = q - head * plane;
    for (int k = 1; k <= n_win; ++k) {
      const double c = (double)p[k - 1];
      const int64_t idx = ((int64_t)head * n_win + (k - 1)) * plane + rem;
      add_f64(img + idx, c);
      if (img2) add_f64(img2 + idx, c * c);
    }
  }
}

// Binned accumulation of many pairs. One FP64 atomic for each pair, window and image goes to memory
// at random (about 25 of them per ns over the chip, 0.9 10^6 pairs x 3 windows x 2 images 257 us), so
// the pairs are first put in order of their pixel's bin (bin_count, bin_scatter: a counting sort
// whose records hold the weighted probabilities), and a workgroup for each bin and window sums its
// 4096 pixels in LDS and adds them to the images. Bins of 4096 pixels:
// two workgroups a CU with both images, and a scattering workgroup's records still run together.
constexpr int BIN_SHIFT = 12, BIN = 1 << BIN_SHIFT, MAX_BINS = 8192;
constexpr int SORT_THREADS = 1024, SORT_PAIRS = 4096;  // pairs per sorting workgroup

// The direct kernel takes 0.044 ns for each atomic (pair, window, image); the binned ones 35 us for
// their four launches, the reading and writing of the image lines that the pairs touch, and 0.65 ns
// for each pair of a bin, which one workgroup per window goes through (15 atomics' time; with few
// bins most of the chip waits for them). Measured with 3 windows of 128 x 128, us direct / binned:
// 16 heads with squares 128000 pairs 37 / 40, 256000 72 / 44, 10^6 267 / 61; 128 heads 128000
// 37 / 60, 256000 72 / 64, 10^6 268 / 86; without squares 16 heads 256000 39 / 40, 10^6 144 / 57,
// 128 heads 256000 39 / 50, 10^6 141 / 69; 10^6 pairs with squares on one head of 64 x 64 (one bin)
// 253 / 688, of 128 x 128 (4 bins) 263 / 202 and with one window 91 / 192, on two of those 92 / 111
// and on four 92 / 70. The line lies a little above where they meet.
bool binned_pays(int64_t m, int64_t n_win, int64_t n_pix, int64_t images) {
  const int64_t bins = (n_pix + BIN - 1) / BIN;
  return m * n_win * images >= (1 << 20) + n_pix * n_win * images / 24 + 15 * m / bins;
}

struct BinWork {
  uint32_t *count;   // pairs of each bin
  uint32_t *cursor;  // of them placed so far
  uint32_t *first;   // first record of each bin, and the end of the last
  float4 *rec;       // per pair quads of (probabilities x weight ..., pixel in bin as bits last)
};

__global__ void __launch_bounds__(256) bin_clear_kernel(uint32_t *p, int n) {
  const int i = (int)(blockIdx.x * 256 + threadIdx.x);
  if (i < n) p[i] = 0u;
}

// pairs of this workgroup in each bin, in LDS
__device__ __forceinline__ void bin_histogram(const int32_t *__restrict__ pix, int64_t lo, int64_t hi, int bins,
                                              uint32_t n_pix, uint32_t *hist) {
  for (int b = (int)threadIdx.x; b < bins; b += SORT_THREADS) hist[b] = 0u;
  __syncthreads();
  for (int64_t r = lo + threadIdx.x; r < hi; r += SORT_THREADS) {
    const uint32_t q = (uint32_t)pix[r];
    if (q < n_pix) atomicAdd(&hist[q >> BIN_SHIFT], 1u);
  }
  __syncthreads();
}

__global__ void __launch_bounds__(SORT_THREADS) bin_count_kernel(const int32_t *__restrict__ pix, int64_t m, int bins,
                                                                 uint32_t n_pix, BinWork W) {
  __shared__ uint32_t hist[MAX_BINS];
  const int64_t lo = (int64_t)blockIdx.x * SORT_PAIRS, hi = min(lo + (int64_t)SORT_PAIRS, m);
  bin_histogram(pix, lo, hi, bins, n_pix, hist);
  for (int b = (int)threadIdx.x; b < bins; b += SORT_THREADS)
    if (hist[b]) atomicAdd(&W.count[b], hist[b]);
}

template <int QUADS>
__global__ void __launch_bounds__(SORT_THREADS) bin_scatter_kernel(const float *__restrict__ logits, int64_t ldl,
                                                                   int64_t m, const int32_t *__restrict__ pix,
                                                                   const float *__restrict__ wgt, int n_win, int bins,
                                                                   uint32_t n_pix, BinWork W) {
  __shared__ uint32_t at[MAX_BINS], first[MAX_BINS];
  __shared__ uint32_t s_wave[SORT_THREADS / 64];
  const int t = (int)threadIdx.x;
  // first record of each bin: every workgroup sums the counts (bins of a thread side by side)
  const int per = (bins + SORT_THREADS - 1) / SORT_THREADS;
  uint32_t mine = 0;
  for (int b = t * per; b < min((t + 1) * per, bins); ++b) mine += W.count[b];
  uint32_t run = mine;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t o = __shfl_up(run, d, 64);
    if ((t & 63) >= d) run += o;
  }
  if ((t & 63) == 63) s_wave[t >> 6] = run;
  __syncthreads();
  uint32_t before = run - mine;
  for (int q = 0; q < (t >> 6); ++q) before += s_wave[q];
  for (int b = t * per; b < min((t + 1) * per, bins); ++b) {
    first[b] = before;
    before += W.count[b];
  }
  const int64_t lo = (int64_t)blockIdx.x * SORT_PAIRS, hi = min(lo + (int64_t)SORT_PAIRS, m);
  bin_histogram(pix, lo, hi, bins, n_pix, at);
  for (int b = t; b < bins; b += SORT_THREADS) {
    if (blockIdx.x == 0) {
      W.first[b] = first[b];
      if (b == bins - 1) W.first[bins] = first[b] + W.count[b];
    }
    if (at[b]) at[b] = first[b] + atomicAdd(&W.cursor[b], at[b]);
  }
  __syncthreads();
  for (int64_t r = lo + t; r < hi; r += SORT_THREADS) {
    const uint32_t q = (uint32_t)pix[r];
    if (q >= n_pix) continue;
    float v[4 * QUADS] = {};
    softmax_row(logits + r * ldl, n_win, wgt[r], v);
    v[4 * QUADS - 1] = __uint_as_float(q & (BIN - 1));
    float4 *out = W.rec + (int64_t)atomicAdd(&at[q >> BIN_SHIFT], 1u) * QUADS;
#pragma unroll
    for (int k = 0; k < QUADS; ++k) out[k] = make_float4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
  }
}

__device__ __forceinline__ void lds_add_f64(double *p, double v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// SHARED: others may add to the images meanwhile, as they may with the direct kernel, so each touched
// pixel takes an atomic (10^6 pairs, 3 windows, squares: 64 heads 71 -> 81 us, 128 heads 86 -> 112).
template <int QUADS, bool SQUARED, bool SHARED>
__global__ void __launch_bounds__(512) bin_accumulate_kernel(BinWork W, int n_win, uint32_t n_pix, int plane,
                                                             double *img, double *img2) {
  __shared__ double sum[SQUARED ? 2 * BIN : BIN];
  const uint32_t lo = W.first[blockIdx.x], hi = W.first[blockIdx.x + 1];
  if (lo == hi) return;
  for (int i = (int)threadIdx.x; i < (SQUARED ? 2 * BIN : BIN); i += 512) sum[i] = 0.0;
  __syncthreads();
  const int k = (int)blockIdx.y;
  const float *rec = (const float *)W.rec;
  for (uint32_t r = lo + threadIdx.x; r < hi; r += 512) {
    const float *v = rec + (int64_t)r * (4 * QUADS);
    const double c = (double)v[k];
    const uint32_t p = __float_as_uint(v[4 * QUADS - 1]);
    lds_add_f64(sum + p, c);
    if (SQUARED) lds_add_f64(sum + BIN + p, c * c);
  }
  __syncthreads();
  for (int i = (int)threadIdx.x; i < BIN; i += 512) {
    const uint32_t q = (uint32_t)blockIdx.x * BIN + (uint32_t)i;
    if (q >= n_pix) break;
    const double s = sum[i], s2 = SQUARED ? sum[BIN + i] : 0.0;
    if (s == 0.0 && s2 == 0.0) continue;
    const uint32_t head = q / (uint32_t)plane, rem = q - head * (uint32_t)plane;
    const int64_t idx = ((int64_t)head * n_win + k) * plane + rem;
    if (SHARED) {
      add_f64(img + idx, s);
      if (SQUARED) add_f64(img2 + idx, s2);
    } else {
      img[idx] += s;
      if (SQUARED) img2[idx] += s2;
    }
  }
}

__global__ void __launch_bounds__(256) counts_accumulate_kernel(const int32_t *__restrict__ cls,
                                                                const int32_t *__restrict__ pix,
                                                                const float *__restrict__ wgt, int64_t m, int n_win,
                                                                int plane, double *img, double *img2) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < m; r += stride) {
    const int c = cls[r];
    if (c <= 0 || c > n_win) continue;
    const int32_t q = pix[r];
    const int32_t head = q / plane, rem = q - head * plane;
    const int64_t idx = ((int64_t)head * n_win + (c - 1)) * plane + rem;
    const double wv = (double)wgt[r];
    add_f64(img + idx, wv);
    if (img2) add_f64(img2 + idx, wv * wv);
  }
}

int grid_for(int64_t n, int per_cu = 16) {
  int dev = 0, n_cu = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
  const int64_t want = (n + 255) / 256;
  return (int)std::max<int64_t>(1, std::min<int64_t>(want, (int64_t)n_cu * per_cu));
}

}  // namespace

extern "C" int gh_spect_pairs(const float *const rec[8], int64_t n, const gh_spect_desc *det, const float *angle_cs,
                              int64_t capacity, void *x16, int32_t *pix, float *wgt, float *const det_rec[8],
                              float *theta_phi, unsigned long long *count, void *stream) {
  if (!rec || !det || !angle_cs || !pix || !wgt || !count || n < 0 || capacity < 0) return GH_EINVAL;
  for (int k = 0; k < 8; ++k)
    if (!rec[k]) return GH_EINVAL;
  if (det->n_proj <= 0 || det->nx <= 0 || det->ny <= 0 || !(det->spacing[0] > 0.0f) || !(det->spacing[1] > 0.0f) ||
      !(det->cos_theta_max > 0.0f && det->cos_theta_max < 1.0f) || !(det->radius > 0.0f) || det->pitch < 0.0f ||
      (int64_t)det->n_proj * det->nx * det->ny > INT32_MAX)
    return GH_EINVAL;
  PairOut o{};
  o.x16 = (__bf16 *)x16; o.pix = pix; o.wgt = wgt; o.tp = theta_phi; o.count = count; o.capacity = capacity;
  if (det_rec) {
    for (int k = 0; k < 8; ++k) {
      if (!det_rec[k]) return GH_EINVAL;
      o.det[k] = det_rec[k];
    }
  }
  if (n == 0) return GH_OK;
  // as many workgroups as the chip holds at once (27 KiB of LDS each, 34 with detector records):
  // each then writes its pairs out few times
  const dim3 grid(grid_for(n, det_rec ? 4 : 5));
  if (det_rec)
    hipLaunchKernelGGL(spect_pairs_kernel<true>, grid, dim3(256), 0, (hipStream_t)stream, rec[0], rec[1], rec[2],
                       rec[3], rec[4], rec[5], rec[6], rec[7], n, *det, angle_cs, o);
  else
    hipLaunchKernelGGL(spect_pairs_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, rec[0], rec[1], rec[2],
                       rec[3], rec[4], rec[5], rec[6], rec[7], n, *det, angle_cs, o);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}

// parameters of a blurring law are finite and give a non-negative width at the law's
// reference point
static bool blur_ok(const gh_blur &B) {
  switch (B.law) {
    case GH_BLUR_NONE: return true;
    case GH_BLUR_GAUSSIAN: return B.sigma >= 0.0f && std::isfinite(B.sigma);
    case GH_BLUR_INVERSE_SQUARE:
      return B.resolution >= 0.0f && std::isfinite(B.resolution) && B.reference > 0.0f && std::isfinite(B.reference);
    case GH_BLUR_LINEAR:
      return B.resolution >= 0.0f && std::isfinite(B.resolution) && B.reference >= 0.0f &&
             std::isfinite(B.reference) && std::isfinite(B.slope);
    default: return false;
  }
}

extern "C" int gh_energy_windows(const float *edep, int64_t n, uint64_t seed, uint64_t first, const gh_blur *blur,
                                 const float *win, int32_t n_win, int32_t *cls, void *stream) {
  if (!edep || !cls || !win || !blur || n < 0 || n_win <= 0 || n_win > MAX_WIN || !blur_ok(*blur))
    return GH_EINVAL;
  Windows W{};
  W.n = n_win;
  for (int k = 0; k < n_win; ++k) {
    W.lo[k] = win[2 * k];
    W.hi[k] = win[2 * k + 1];
    if (!(W.hi[k] > W.lo[k])) return GH_EINVAL;
  }
  if (n == 0) return GH_OK;
  hipLaunchKernelGGL(energy_windows_kernel, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, edep, n,
                     (uint32_t)seed, (uint32_t)(seed >> 32), first, *blur, W, cls);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}

extern "C" int gh_arf_accumulate(const float *logits, int64_t ldl, int64_t m, const int32_t *pix, const float *wgt,
                                 int32_t n_win, int32_t plane, double *img, double *img2, void *stream) {
  if (!logits || !pix || !wgt || !img || m < 0 || n_win <= 0 || n_win > MAX_WIN || ldl < n_win + 1 || plane <= 0)
    return GH_EINVAL;
  if (m == 0) return GH_OK;
  hipLaunchKernelGGL(arf_accumulate_kernel, dim3(grid_for(m)), dim3(256), 0, (hipStream_t)stream, logits, ldl, m, pix,
                     wgt, (int)n_win, (int)plane, img, img2);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}

namespace {

int bin_quads(int32_t n_win) { return (n_win + 4) / 4; }

int64_t bin_head_words(int64_t bins) { return (3 * bins + 1 + 3) / 4 * 4; }  // count, cursor, first

template <int QUADS, bool SHARED>
void launch_binned(const float *logits, int64_t ldl, int64_t m, const int32_t *pix, const float *wgt, int n_win,
                   int plane, int bins, uint32_t n_pix, BinWork W, double *img, double *img2, hipStream_t st) {
  const dim3 sort((unsigned)((m + SORT_PAIRS - 1) / SORT_PAIRS));
  hipLaunchKernelGGL(bin_clear_kernel, dim3((2 * bins + 255) / 256), dim3(256), 0, st, W.count, 2 * bins);
  hipLaunchKernelGGL(bin_count_kernel, sort, dim3(SORT_THREADS), 0, st, pix, m, bins, n_pix, W);
  hipLaunchKernelGGL(bin_scatter_kernel<QUADS>, sort, dim3(SORT_THREADS), 0, st, logits, ldl, m, pix, wgt, n_win, bins,
                     n_pix, W);
  if (img2)
    hipLaunchKernelGGL((bin_accumulate_kernel<QUADS, true, SHARED>), dim3(bins, n_win), dim3(512), 0, st, W, n_win,
                       n_pix, plane, img, img2);
  else
    hipLaunchKernelGGL((bin_accumulate_kernel<QUADS, false, SHARED>), dim3(bins, n_win), dim3(512), 0, st, W, n_win,
                       n_pix, plane, img, img2);
}

template <bool SHARED>
int accumulate_binned(const float *logits, int64_t ldl, int64_t m, const int32_t *pix, const float *wgt, int32_t n_win,
                      int32_t plane, int64_t n_pix, double *img, double *img2, void *work, int64_t work_bytes,
                      void *stream) {
  if (!logits || !pix || !wgt || !img || !work || m < 0 || m > INT32_MAX || n_win <= 0 || n_win > MAX_WIN ||
      ldl < n_win + 1 || plane <= 0 || n_pix <= 0 || n_pix > INT32_MAX || ((uintptr_t)work & 15) != 0)
    return GH_EINVAL;
  const int64_t bins = (n_pix + BIN - 1) / BIN;
  if (bins > MAX_BINS || work_bytes < 4 * bin_head_words(bins) + 16 * bin_quads(n_win) * m) return GH_EINVAL;
  if (m == 0) return GH_OK;
  uint32_t *w = (uint32_t *)work;
  const BinWork W{w, w + bins, w + 2 * bins, (float4 *)(w + bin_head_words(bins))};
  const hipStream_t st = (hipStream_t)stream;
  const auto launch = bin_quads(n_win) == 1 ? launch_binned<1, SHARED> :
                      bin_quads(n_win) == 2 ? launch_binned<2, SHARED> : launch_binned<3, SHARED>;
  launch(logits, ldl, m, pix, wgt, n_win, plane, (int)bins, (uint32_t)n_pix, W, img, img2, st);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}

}  // namespace

extern "C" int gh_arf_accumulate_workspace(int64_t m, int32_t n_win, int64_t n_pix, int32_t squared, int64_t *bytes) {
  if (!bytes || m < 0 || n_win <= 0 || n_win > MAX_WIN || n_pix < 0) return GH_EINVAL;
  const int64_t bins = (n_pix + BIN - 1) / BIN;
  *bytes = 0;
  if (bins == 0 || bins > MAX_BINS || m > INT32_MAX || !binned_pays(m, n_win, n_pix, squared ? 2 : 1)) return GH_OK;
  *bytes = 4 * bin_head_words(bins) + 16 * bin_quads(n_win) * m;
  return GH_OK;
}

extern "C" int gh_arf_accumulate_binned(const float *logits, int64_t ldl, int64_t m, const int32_t *pix,
                                        const float *wgt, int32_t n_win, int32_t plane, int64_t n_pix, double *img,
                                        double *img2, void *work, int64_t work_bytes, void *stream) {
  return accumulate_binned<true>(logits, ldl, m, pix, wgt, n_win, plane, n_pix, img, img2, work, work_bytes, stream);
}

extern "C" int gh_arf_accumulate_binned_own(const float *logits, int64_t ldl, int64_t m, const int32_t *pix,
                                            const float *wgt, int32_t n_win, int32_t plane, int64_t n_pix, double *img,
                                            double *img2, void *work, int64_t work_bytes, void *stream) {
  return accumulate_binned<false>(logits, ldl, m, pix, wgt, n_win, plane, n_pix, img, img2, work, work_bytes, stream);
}

extern "C" int gh_counts_accumulate(const int32_t *cls, const int32_t *pix, const float *wgt, int64_t m, int32_t n_win,
                                    int32_t plane, double *img, double *img2, void *stream) {
  if (!cls || !pix || !wgt || !img || m < 0 || n_win <= 0 || n_win > MAX_WIN || plane <= 0) return GH_EINVAL;
  if (m == 0) return GH_OK;
  hipLaunchKernelGGL(counts_accumulate_kernel, dim3(grid_for(m)), dim3(256), 0, (hipStream_t)stream, cls, pix, wgt, m,
                     (int)n_win, (int)plane, img, img2);
  return hipGetLastError() == hipSuccess ? GH_OK : GH_EHIP;
}
