// The propagator W <- P E6(V) P W (afqmc_sys::propagate,
// src/AFQMC/afqmc_sys.hpp:146-173, with apply_expM, src/AFQMC/vHS.hpp:61-91,
// summed by Horner's rule) of small systems as one kernel.
#pragma once
#include "common.hpp"

struct PropSmallArgs {
  zd* W;          // [nw][2][M][N], updated in place
  const void* P;  // [M][M] Propg1 in the contraction format (zd, zf or zb)
  const void* V;  // [nw][M][M] HS potential, the same format
  int M, N, nw;
  int ncb;        // column blocks per walker, ceil(2N / NB)
};

// largest M per contraction format: M / 16 waves hold the left operand
constexpr int PS_MMAX = 192;      // FP32 and split-BF16
constexpr int PS_MMAX_F64 = 128;  // FP64

// format: 0 zd, 1 zf, 2 zb
bool prop_small_ok(int mode_format, int M);  // whether it has a kernel for M
void prop_small_launch(hipStream_t st, PropSmallArgs a, int mode_format);
