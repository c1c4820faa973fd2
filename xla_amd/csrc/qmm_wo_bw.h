// Arguments and launchers of the weight-only tiled GEMM for blockwise and int4 weights
// (qmm_wo_gemm_bw.hip), called from the workspace entry point in qmm_wo_gemm.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#include "qmm_common.h"

struct WoBwArgs {
  const void* x;      // [M, K], bf16 or f16
  const uint8_t* w;   // tiled weight, 8 or 4 bits
  const void* scale;  // [K/C, N] of x's dtype
  const void* zp;     // [K/C, N] of x's dtype, or null
  void* out;          // [M, N] of x's dtype
  int M, N, K, C;     // C: columns per quantization block (K for per-channel weights)
};

// bits = 4 or 8; x's dtype by launcher
int qmm_wo_bw_launch_bf16(const WoBwArgs& a, int bits, hipStream_t stream);
int qmm_wo_bw_launch_f16(const WoBwArgs& a, int bits, hipStream_t stream);
// the same in tiles of 64 x 256 (qmm_wo_gemm_bw_wide.hip), called by the launchers above; cus: compute units to fill;
// a zero point only with bits = 4 and C = 128
int qmm_wo_bw_wide_launch_bf16(const WoBwArgs& a, int bits, int cus, hipStream_t stream);
int qmm_wo_bw_wide_launch_f16(const WoBwArgs& a, int bits, int cus, hipStream_t stream);

// Two dot products rounded to x's dtype, as f32.  bf16: one at a time, beside a zero, which leaves the value in f32 (as a
// pair and unpacked again it is three instructions for two; 2048 x 4096 x 4096 int4 in blocks of 128 with zero points:
// 80.5 -> 77.0 us).  f16: as a pair (one at a time 77.1 -> 81.4).
template <int XT> __device__ __forceinline__ void wo_bw_round2(float d0, float d1, float& p0, float& p1) {
  if constexpr (XT == XLA_AMD_DT_BF16) {
    p0 = qmm_round_dt(d0, XT);
    p1 = qmm_round_dt(d1, XT);
  } else {
    const uint32_t p = qmm_f32x2_to_f16x2(d0, d1);
    p0 = qmm_from_raw(p & 0xffffu, XT);
    p1 = qmm_from_raw(p >> 16, XT);
  }
}
