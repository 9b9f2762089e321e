// Host-side declarations of the weight-gradient kernels (frnn_grad_gemm.hip).
#pragma once
#include "frnn_common.h"

namespace frnn {

struct GradGemmArgs {
  const void* gsrc[4];   // per recurrent gate g: cotangent of its pre-activation; element
                         // (row r = b*T + t, head n, unit d) at gsrc[g] + r*gld[g] + n*D + d
  long gld[4];           // row strides in elements
  const void* states_h;  // h of all steps, [B,T,N,D] (state 0 of the states tensor)
  const void* s0_h;      // initial h, [B,N,D]
  float* part;           // [splits][G_r][N][D][D] partial sums
  int B, T, N, D, GR;
  int rows_per_split;    // filled in by launch_grad_gemm
  // one split: the GEMM's sums are dR itself, and its workgroups also sum the bias partials
  void* dR;              // null: not here (the sums go to part)
  const float* part_b;   // [splits_b][n_b]
  int splits_b; long n_b;
  void* db;
  int narrow;            // 1: dR, 2: db in the 16-bit storage type (of the kernel), else fp32
};

// Rt = R transposed per head; zero_bytes > 0: the same launch clears that many bytes at `zero` (16-byte aligned, whole words)
int launch_transpose_r(int dtype, const void* R, void* Rt, int N, int D, int GR, hipStream_t st, void* zero = nullptr, size_t zero_bytes = 0);
int grad_gemm_splits(int dtype, int B, int T, int N, int D, int GR);
int launch_grad_gemm(int dtype, GradGemmArgs a, int splits, hipStream_t st);
// narrow: 1: dR, 2: db in the storage type `dtype`, else fp32
int launch_grad_reduce(int dtype, int narrow, const float* part_r, int splits_r, size_t n_r, void* dR,
                       const float* part_b, int splits_b, size_t n_b, void* db, hipStream_t st);
// (a second block may be cleared by the same launch)
int launch_fill_zero(void* p, size_t bytes, hipStream_t st, void* p2 = nullptr, size_t bytes2 = 0);

}  // namespace frnn
