// Split-K plan of a BF16 GEMM, shared by gh_gemm_bf16 and the fused weight gradients.
#pragma once
#include <algorithm>

#include "../../include/gatehip.h"

namespace gh {

constexpr int GEMM_BM = 64, GEMM_BN = 64, GEMM_BK = 32;

// S slices of kc (a multiple of GEMM_BK) reduction elements each; S = 1 means no split. Weight
// gradients (few output tiles, long reduction) are split so that the launch fills the chip;
// the slices are then summed in a fixed order.
inline void splitk_plan(int M, int N, int K, int mode, int &S, int &kc) {
  const int tiles = ((N + GEMM_BN - 1) / GEMM_BN) * ((M + GEMM_BM - 1) / GEMM_BM);
  S = 1;
  kc = ((K + GEMM_BK - 1) / GEMM_BK) * GEMM_BK;
  if (mode == GH_EPI_STORE && tiles < 512 && K >= 2048) {
    S = std::max(1, std::min((K + 511) / 512, std::max(1, 1024 / tiles)));
    kc = (K + S - 1) / S;
    kc = (kc + GEMM_BK - 1) / GEMM_BK * GEMM_BK;
    S = (K + kc - 1) / kc;
  }
}

}  // namespace gh
