// fqa_gemm_internal.h — the projection GEMM as a building block of fused entry points.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fqa {

// The norm / RoPE / append a QKV projection's epilogue applies when it runs unsplit
// (the arguments of fqa_qknorm_rope_append).
struct GemmAppend {
  const float* wq;
  const float* wk;
  const float* cos_tab;
  const float* sin_tab;
  int rope_max_pos;
  const int32_t* positions;
  const int32_t* slots;
  const int32_t* meta;
  uint16_t* pool;
  long long pool_pages;
  float eps;
  int write_k;
};

// The QKV projection x . W^T (N = 6144, y = the qkv buffer) with fqa_gemm's argument rules
// and plan, for a caller that appends.  An unsplit plan on the 128- and 256-row tiles applies
// `app` (the per-head norm + RoPE + paged append) in its epilogue, with the results
// fqa_qknorm_rope_append would give on fqa_gemm's y; *appended says so.  Otherwise the fp32
// partials land in `workspace` as [planes][M][N], to be summed in plane order as fqa_gemm's
// reduction does, and y is not written.  Returns the number of planes, 0 for M = 0 or when
// appended, or an FQA_E code.
int gemm_launch_partials(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y,
                         int64_t ldy, int32_t M, int32_t N, int32_t K, void* workspace,
                         int64_t workspace_bytes, hipStream_t st,
                         const GemmAppend& app, bool* appended);

}  // namespace fqa
