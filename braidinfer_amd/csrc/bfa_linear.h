// The linear-layer kernels that bfa_linear (qkv.hip) launches: the GEMM for 65 and
// more tokens (linear_gemm.hip) and the one-launch weight stream for few
// (linear_gemv.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bfa_gemm_plan.h"

namespace bfa {

// y = out_dt(mid_dt(proj_dt(x W^T + bias) + res)), or with swiglu
// out_dt(proj_dt(silu(proj_dt(gate))) * proj_dt(up)).  x and W share a 16-bit
// dtype, rows 16-byte aligned, k a multiple of 64, byte offsets of x and W
// below 4 GiB.
struct LinArgs {
  const uint16_t* a;  // x [m, k]
  const uint16_t* w;  // W [n, k], or [2 n, k] gate rows then up rows
  int64_t m, n, k, lda, ldw;
  const void* bias;  // [n], plain only
  const void* res;   // [m, n], plain only
  void* out;
  int64_t ldr, ldo;
  int bias_dt, res_dt, proj_dt, mid_dt, out_dt;
  int vec;  // res and out take 16-byte accesses at multiples of 8 columns
  int swiglu;
  float* part;  // split-K partial tiles
  // (set by the launcher)
  int tiles_m, tiles_n, full, splits, kt;
  int pairs;  // out takes 4-byte stores at even columns
};

// The plan for m tokens and n output columns (2 n weight rows with swiglu);
// split = false: without split K, so without a workspace.
GemmPlan linear_plan(int64_t m, int64_t n, int64_t k, bool swiglu, bool split);
void launch_linear_gemm(const GemmPlan& p, LinArgs q, int dt, hipStream_t st);

// One launch, no workspace (of LinArgs: part and the planner's fields unused);
// splits: of the split-K kernels for the same call.
bool linear_gemv_ok(int64_t m, int64_t wrows, int64_t k, bool swiglu, int64_t splits);
void launch_linear_gemv(LinArgs q, int dt, hipStream_t st);

}  // namespace bfa
