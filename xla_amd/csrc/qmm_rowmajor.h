// Arguments and launcher of the matmul against a row-major int8 weight (qmm_rowmajor.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

struct QmmRowMajorArgs {
  const void* x;       // [M, K] of x's dtype, or int8
  const int8_t* w;     // [N, K]
  const void* scale;   // [N] weight scale
  const void* zp;      // [N] or null
  void* out;           // [M, N]
  int64_t M, N, K;
  int scale_dt, zp_dt, zpo_dt, out_dt;
  int dot_dt, store_dt;               // weight-only
  const void* x_scale;                // int8 activations: [M]
  const int32_t* x_sum;               // ... [M], with a zero point
  int32_t* acc_out;                   // ... raw sums, or null
  int x_scale_dt, cvt_dt, mid_dt;
  int64_t ldo;         // elements between rows of out (and acc_out): N, or more in a piece of the channels
};

constexpr int kQmmRowMajorInt8 = 3;  // x_dt of int8 activations
int qmm_rowmajor_launch(const QmmRowMajorArgs& a, int x_dt, hipStream_t stream);
