// LM head for 33 to 256 token rows (csrc/lm_head_wide.hip).
#pragma once

#include "common.h"

namespace oxr {

constexpr int kWideMaxGrid = 1024;  // bound on the workgroups (sizes the workspace)
constexpr int kWideMaxRows = 256;

// Per workgroup t < grid and row m: the key (largest bf16 logit, then lowest column) of its columns at
// best[t * M + m]; bf16 logits [M, N] too unless null.  xp: the token rows packed; w: the packed weight;
// K a multiple of 128.  grid is at most the number of 32-row vocab tiles.
int launch_lm_head_wide(const bf16_t* xp, int M, const bf16_t* w, int64_t K, int64_t N, bf16_t* logits,
                        uint64_t* best, int grid, hipStream_t s);

}  // namespace oxr
