// Tiled bf16 GEMM for more than 64 token rows (csrc/gemm_tile.hip).
#pragma once

#include "common.h"

namespace oxr {

// Y = X * W^T over token rows [0, m) and output columns [0, n); epilogues as in csrc/gemm.hip.
struct TileArgs {
  const bf16_t* x;   // [m, ldx] row-major, or packed (ldx = k)
  int64_t ldx;
  int64_t m;
  const bf16_t* w;   // [rows, k] row-major, or packed
  int64_t k;
  int64_t n;         // output columns (gate rows for kSiluMul)
  bf16_t* y;         // [m, ldy], or packed with row length n
  int64_t ldy;
  float* part;       // kPartial: [k_splits, m, n]
  int k_splits;
  bool x_packed, w_packed, y_packed;
};

// Whether the kernel's offsets and grid hold these sizes.
bool gemm_tile_supported(const TileArgs& a);

// epilogue: 0 store, 1 SiLU * mul, 3 add to y, 4 fp32 partial sums.  Operands are checked by the caller.
// The k slice is summed as `parts` partial sums added in order (each a multiple of 128 long), or as one chain.
int launch_gemm_tile(const TileArgs& a, int epilogue, int parts, bool one_chain, hipStream_t s);

}  // namespace oxr
