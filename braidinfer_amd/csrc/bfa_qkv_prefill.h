// The QKV projection above 64 tokens for head_dim 64 and 128 (qkv_prefill.hip),
// launched by the QKV entry points (qkv.hip).
#pragma once

#include "bfa_gemm_plan.h"
#include "bfa_qkv.h"

namespace bfa {

struct QkvPrefillArgs {
  const uint16_t* a;  // operand [m, k]
  const uint16_t* w;  // weight [e.n, k]
  int64_t m, k, lda, ldw;
  float* part;  // split-K partial tiles
  // (set by the launcher)
  int tiles_m, tiles_n, full, splits, kt;
  int vec_out, vec_cache, stream;
};

// The plan for m tokens and n columns; split = false: without split K, so
// without a workspace for partials.
GemmPlan qkv_prefill_plan(int64_t m, int64_t n, int64_t k, int64_t operand_bytes, bool split);
// dt: operand and weight (bf16 or fp16), k a multiple of 64, rows 16-byte
// aligned, byte offsets of either below 4 GiB; edt: the epilogue's dtype form.
void launch_qkv_prefill(const GemmPlan& p, QkvPrefillArgs q, const QkvEpi& e, int dt, int edt, hipStream_t st);

}  // namespace bfa
