// Host-side declarations of the single-step kernel of the fused backend (frnn_step.hip).
#pragma once
#include "frnn_common.h"
#include "frnn_plan.h"

namespace frnn {

struct StepArgs {
  const void* Wx; const void* R; const void* b; const void* s0; void* states;
  float* carry;    // [S][B][N][D] fp32, or null: see FwdArgs
  int B, BS, N, D;
  float h_clip;
  // the order in which the sequence kernel of this size sums over k (set by launch_fused_step)
  int own_ks, ut_wg;  // k-steps of a workgroup's own slice where those come first (0: k in order), unit tiles per workgroup
  int ksp, nacc;      // parts of k that are summed apart; chains that take turns over k (one-gate cells)
  int bias_first;     // the bias starts the first chain (16-row tiles) or is added to the sum
};

// 16-bit types; p and tile_rows: the tiling of a sequence call of this size
int launch_fused_step(int function, int dtype, const Plan& p, int tile_rows, StepArgs a, hipStream_t st);

}  // namespace frnn
