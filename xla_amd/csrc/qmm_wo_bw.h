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

// ---- K split over the waves of a workgroup (qmm_wo_ksplit_bw.hip) ----
// Tiles of that kernel: rows, channels, K groups of waves, whether it takes a zero point, and two estimates of a launch's
// time, us, from rounds of 256 tiles and steps of 128 columns per wave (whole blocks).
// The first picks the tile; fitted to 78 - 185 measured launches per tile (8 - 1000 rows, 18 weights of N 512 - 14336, K
// 1024 - 14336, 4 and 8 bits; root mean square error 7 - 11 %):
//   fixed + round * rounds + (step + zp (with a zero point) + int8 (8 bits)) * rounds * steps + load * tiles / 256 * steps
//     + weight * (bytes of the weight) / 10^6
// The second, with the blocks' ends, says whether the launch takes it at all; fitted to 12000 - 24000 launches per tile
// (17 - 1000 rows, N 256 - 16384, K 512 - 14336, blocks of 128 - 1024 columns and per channel, weights out of HBM; error
// 6 - 10 %, 5.5 % of the larger tiles):
//   fixed + round * rounds + (step + int8 (8 bits) + perch (per channel)) * rounds * steps + load * tiles / 256 * steps
//     + (block + zp (with a zero point)) * rounds * (blocks per wave) + weight * (bytes of the weight) / 10^6
struct KsBwTile {
  uint32_t bm, bn, kw;
  bool with_zp;
  float fixed, round, step, load, weight, zp, int8;
  struct {
    float fixed, round, step, load, weight, block, zp, int8, perch;
  } time;
};
constexpr KsBwTile kKsBwTiles[] = {
    {16, 16, 8, true, 2.46f, 0.10f, 0.681f, 0.252f, 0.032f, 0.185f, 0.197f,
     {3.411f, 0.074f, 0.811f, 0.186f, 0.016f, -0.132f, 0.121f, 0.012f, -0.337f}},
    {16, 32, 8, true, 1.72f, 1.08f, 0.906f, 0.130f, 0.080f, 0.282f, 0.231f,
     {2.681f, 0.863f, 0.969f, 0.177f, 0.017f, -0.093f, 0.253f, 0.089f, -0.398f}},
    {32, 32, 4, true, 1.62f, 1.67f, 0.648f, 0.116f, 0.061f, 0.189f, -0.036f,
     {2.571f, 1.045f, 0.723f, 0.130f, 0.017f, -0.032f, 0.135f, -0.038f, -0.170f}},
    {48, 32, 4, true, 1.46f, 1.87f, 0.748f, 0.091f, 0.103f, 0.267f, 0.008f,
     {1.896f, 1.699f, 0.757f, 0.125f, 0.033f, 0.095f, 0.206f, -0.011f, -0.135f}},
    {48, 64, 4, true, 0.95f, 2.90f, 1.034f, 0.085f, 0.083f, 0.351f, -0.026f,
     {1.523f, 2.349f, 0.985f, 0.172f, 0.025f, 0.180f, 0.293f, -0.023f, -0.073f}},
    {64, 32, 4, true, 1.43f, 2.12f, 0.819f, 0.188f, 0.069f, 0.258f, -0.054f,
     {1.813f, 1.728f, 0.852f, 0.257f, -0.027f, 0.045f, 0.206f, -0.013f, -0.110f}},
    {64, 64, 4, false, 0.64f, 3.27f, 1.200f, 0.167f, 0.074f, 0.000f, -0.077f,
     {1.322f, 2.215f, 1.113f, 0.235f, 0.020f, 0.320f, 0.000f, -0.138f, -0.035f}},
};
// The tile a launch of M rows runs with (-1: not one for this kernel): bf16 or f16 (f16) x and every other dtype x's,
// blockwise (C < K, C % 128 == 0) or int4 weights, N % 4 == 0.  k_slices: in how many slices of k_per_slice columns the
// streaming kernel would run it (1: whole).
int qmm_wo_ksplit_bw_tile(int64_t M, int64_t N, int64_t K, int64_t C, int bits, bool zp, bool f16, int k_slices, int k_per_slice);
int qmm_wo_ksplit_bw_run(int tile, const WoBwArgs& a, int bits, int x_dt, hipStream_t stream);
int qmm_wo_ksplit_bw_launch_bf16_4(const WoBwArgs& a, int tile, hipStream_t stream);
int qmm_wo_ksplit_bw_launch_bf16_8(const WoBwArgs& a, int tile, hipStream_t stream);
int qmm_wo_ksplit_bw_launch_f16_4(const WoBwArgs& a, int tile, hipStream_t stream);
int qmm_wo_ksplit_bw_launch_f16_8(const WoBwArgs& a, int tile, hipStream_t stream);

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
