// Arguments and epilogue shared by the weight-only GEMM kernels (qmm_wo_gemm.hip, qmm_wo_ksplit.hip).
#pragma once
#include "qmm_common.h"

struct WoGemmArgs {
  const void* x;       // [M, K]
  const uint8_t* w;    // tiled weight, 8 bits
  const void* scale;   // [N]
  const void* zp;      // [N] or null
  void* out;           // [M, N] of store_dt (split == 1)
  float* part;         // [split][M][N] partial dot products (split > 1)
  float* part_xs;      // [split][M] partial row sums of x (split > 1, zero point)
  int M, N, K;
  int G;               // channels per group of the tiled weight (xla_amd_qmm_tile_group)
  int k_per_split;     // columns per K slice (a multiple of 128)
  int split;
  int scale_dt, zp_dt, dot_dt, out_dt, store_dt;
  int Kw;    // columns of the weight: K, or K / 3 when x is an f32 matrix split into three bf16 parts side by side
  int x_dt;  // the caller's x dtype (the row sums of x are rounded to it): the kernel's, or f32 for split f32 rows
  int stage_out;  // 128 x 256 tile: results leave through LDS, written out by the copying waves during the next item
};

// The dtypes of the epilogue: those of the call, or (UNI) all equal to x's dtype and known at
// compile time, which is the common case and removes every branch on a dtype.
template <int XT, bool UNI> struct WoDts {
  int scale_dt, zp_dt, dot_dt, out_dt, store_dt, x_dt;
  template <class Args>
  __device__ __forceinline__ explicit WoDts(const Args& a)
      : scale_dt(UNI ? XT : a.scale_dt), zp_dt(UNI ? XT : a.zp_dt), dot_dt(UNI ? XT : a.dot_dt),
        out_dt(UNI ? XT : a.out_dt), store_dt(UNI ? XT : a.store_dt), x_dt(UNI ? XT : a.x_dt) {}
};

// Scale (or zero point) of four consecutive channels as raw bits; channels past N repeat the last one.
__device__ __forceinline__ void wo_load4_raw(const void* p, int n, int N, int dt, uint32_t raw[4]) {
#pragma unroll
  for (int v = 0; v < 4; ++v) raw[v] = qmm_load_raw(p, min(n + v, N - 1), dt);
}

// The reference's epilogue for four consecutive channels of one row:
//   p = round_dot(dot); r = round_out(scale * p); with a zero point r = round_out(r - round_zpo(round_x(xsum) * zp)).
template <class Dts>
__device__ __forceinline__ void wo_finish4_f(const Dts& d, const float* scale, const float* zp, bool has_zp, f32x4 dot,
                                             float xsum, int x_dt, float o[4]) {
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const float p = qmm_round_dt(dot[v], d.dot_dt);
    float r = qmm_round_dt(scale[v] * p, d.out_dt);
    if (has_zp) {
      const int zpo_dt = qmm_promote(x_dt, d.zp_dt);
      const float z = qmm_round_dt(qmm_round_dt(xsum, x_dt) * zp[v], zpo_dt);
      r = qmm_round_dt(r - z, d.out_dt);
    }
    o[v] = r;
  }
}
// ... with scales and zero points as raw bits.
template <class Dts>
__device__ __forceinline__ void wo_finish4(const Dts& d, const uint32_t sraw[4], const uint32_t zraw[4], bool has_zp,
                                           f32x4 dot, float xsum, int x_dt, float o[4]) {
  float s[4], z[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    s[v] = qmm_from_raw(sraw[v], d.scale_dt);
    if (has_zp) z[v] = qmm_from_raw(zraw[v], d.zp_dt);
  }
  wo_finish4_f(d, s, z, has_zp, dot, xsum, x_dt, o);
}

// Stores four consecutive channels of row m starting at channel n (n % 4 == 0).  VEC: N is a
// multiple of 4, so the four channels exist and their address is aligned for one store.
template <bool VEC>
__device__ __forceinline__ void wo_store4(void* out, int m, int n, int N, const float o[4], int store_dt) {
  const size_t idx = (size_t)m * N + n;
  if constexpr (VEC) {
    if (store_dt == XLA_AMD_DT_F32) {
      *(f32x4*)((float*)out + idx) = f32x4{o[0], o[1], o[2], o[3]};
    } else {
      const bool bf = store_dt == XLA_AMD_DT_BF16;
      const uint32_t lo = bf ? qmm_f32x2_to_bf16x2(o[0], o[1]) : qmm_f32x2_to_f16x2(o[0], o[1]);
      const uint32_t hi = bf ? qmm_f32x2_to_bf16x2(o[2], o[3]) : qmm_f32x2_to_f16x2(o[2], o[3]);
      *(i32x2*)((uint16_t*)out + idx) = i32x2{(int)lo, (int)hi};
    }
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (n + v < N) qmm_store(out, idx + v, o[v], store_dt);
  }
}

// Stores the first cnt (1 .. 4) of four consecutive channels of row m starting at channel n, n even: in
// pairs where the row length allows it (rows whose length is no multiple of 4).
__device__ __forceinline__ void wo_store_some(void* out, int m, int n, int N, int cnt, const float o[4], int store_dt) {
  const size_t idx = (size_t)m * N + n;
  if ((N & 1) == 0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (cnt >= 2 * h + 2) {
        if (store_dt == XLA_AMD_DT_F32) {
          typedef float f32x2_t __attribute__((ext_vector_type(2)));
          *(f32x2_t*)((float*)out + idx + 2 * h) = f32x2_t{o[2 * h], o[2 * h + 1]};
        } else {
          *(uint32_t*)((uint16_t*)out + idx + 2 * h) = store_dt == XLA_AMD_DT_BF16 ? qmm_f32x2_to_bf16x2(o[2 * h], o[2 * h + 1])
                                                                                  : qmm_f32x2_to_f16x2(o[2 * h], o[2 * h + 1]);
        }
      } else if (cnt == 2 * h + 1) {
        qmm_store(out, idx + 2 * h, o[2 * h], store_dt);
      }
    }
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (v < cnt) qmm_store(out, idx + v, o[v], store_dt);
  }
}

// The same epilogue and store when every dtype is bf16 and there is no zero point: two
// values per conversion, and the rounded product is already the stored bit pattern.
__device__ __forceinline__ void wo_finish_pack_bf16(const uint32_t sraw[4], f32x4 dot, uint32_t res[2]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t p = qmm_f32x2_to_bf16x2(dot[2 * h], dot[2 * h + 1]);
    const float p0 = __uint_as_float(p << 16), p1 = __uint_as_float(p & 0xffff0000u);
    res[h] = qmm_f32x2_to_bf16x2(__uint_as_float(sraw[2 * h] << 16) * p0, __uint_as_float(sraw[2 * h + 1] << 16) * p1);
  }
}
__device__ __forceinline__ void wo_finish_store_bf16(void* out, int m, int n, int N, const uint32_t sraw[4], f32x4 dot) {
  uint32_t res[2];
  wo_finish_pack_bf16(sraw, dot, res);
  *(i32x2*)((uint16_t*)out + (size_t)m * N + n) = i32x2{(int)res[0], (int)res[1]};
}

// ---- K split over the waves of a workgroup (qmm_wo_ksplit.hip) ----
// Tiles of that kernel: rows, channels, K groups of waves, and the time of a launch, us, as fitted to 111 - 256
// measured shapes per tile (5 - 1024 rows, 24 pairs of N 512 - 28672 and K 512 - 14336, the geometric mean of weights
// out of HBM and out of the Infinity Cache; root mean square error 4 - 8 %):
//   fixed + round * rounds + (step * rounds + load * tiles / 256) * steps + weight * N K / 10^6
// rounds of 256 tiles, steps of 128 columns per wave.
struct KsTile {
  uint32_t bm, bn, kw;
  float fixed, step, load, round, weight;
};
constexpr KsTile kKsTiles[] = {
    {16, 16, 8, 2.66f, 0.498f, 0.195f, 0.415f, 0.046f}, {16, 32, 8, 2.66f, 0.695f, 0.246f, 0.560f, 0.057f},
    {32, 32, 4, 2.32f, 0.545f, 0.140f, 0.888f, 0.027f}, {32, 64, 4, 2.43f, 0.739f, 0.206f, 1.001f, 0.052f},
    {48, 32, 4, 1.82f, 0.575f, 0.149f, 1.805f, 0.036f}, {48, 64, 4, 1.85f, 0.837f, 0.199f, 2.087f, 0.048f},
    {64, 64, 4, 1.40f, 0.962f, 0.344f, 2.313f, 0.031f}, {64, 96, 4, 1.65f, 1.148f, 0.466f, 2.839f, 0.047f},
    {64, 128, 4, 1.54f, 1.337f, 0.672f, 3.471f, 0.041f},
};
// ... and for f32 x: 1036 measurements of 300 shapes with 1 - 127 rows, root mean square error 2 - 8 %.
constexpr KsTile kKsTilesF32[] = {
    {16, 16, 8, 2.66f, 1.323f, 0.269f, 0.406f, 0.009f}, {16, 32, 8, 3.01f, 2.346f, 0.380f, 0.015f, 0.057f},
    {16, 64, 8, 2.16f, 4.711f, 0.129f, 1.077f, 0.078f}, {16, 16, 4, 2.93f, 0.935f, 0.138f, 0.000f, 0.000f},
    {32, 32, 4, 2.46f, 2.119f, 0.207f, 0.919f, 0.022f}, {32, 64, 4, 2.58f, 4.150f, 0.132f, 0.960f, 0.046f},
};
// Arguments of the kernel, tiles included: one struct of no more bytes than the kernel reads.  (A launch's arguments are
// written out by the host each time; with WoGemmArgs, the tiles beside it and the 256 bytes of hidden arguments that
// reading gridDim brings, 392 bytes in all, an eager call of 8 x 1024 x 1024 f32 took 0.1 - 0.15 us longer, of 7.6.)
struct KsTiles {
  int rows, tiles_m, tiles, per_xcd;  // rows per tile (M spread evenly over the row tiles), row tiles, all tiles, tiles per XCD
  uint64_t tiles_m_magic;             // ceil(2^32 / tiles_m)
};
struct KsArgs {
  const void* x;       // [M, K]
  const uint8_t* w;    // tiled weight, 8 bits
  const void* scale;   // [N]
  const void* zp;      // [N] or null
  void* out;           // [M, N] of store_dt
  int M, N, K;
  int G;               // channels per group of the tiled weight (xla_amd_qmm_tile_group)
  int scale_dt, zp_dt, dot_dt, out_dt, store_dt, x_dt;
  KsTiles t;
};
// The tile a launch of M rows of 2-byte x against a per-channel int8 weight runs with (-1: not one for this kernel).
int qmm_wo_ksplit_tile(int64_t M, int64_t N, int64_t K);
// ... of f32 x
int qmm_wo_ksplit_f32_tile(int64_t M, int64_t N, int64_t K);
// Runs a launch with the tile that one of them gave (arguments checked by the entry points: per-channel int8 weight, a tile for it).
int qmm_wo_ksplit_run(int tile, const void* x, const void* w_tiled, const void* scale, const void* zp, void* out, int64_t M, int64_t N,
                      int64_t K, int x_dt, int scale_dt, int zp_dt, int dot_dt, int out_dt, int store_dt, hipStream_t s);
int qmm_wo_ksplit_launch_bf16_0(KsArgs& a, int tile, hipStream_t stream);
int qmm_wo_ksplit_launch_bf16_1(KsArgs& a, int tile, hipStream_t stream);
int qmm_wo_ksplit_launch_bf16_2(KsArgs& a, int tile, hipStream_t stream);
int qmm_wo_ksplit_launch_f16_0(KsArgs& a, int tile, hipStream_t stream);
int qmm_wo_ksplit_launch_f16_1(KsArgs& a, int tile, hipStream_t stream);
int qmm_wo_ksplit_launch_f16_2(KsArgs& a, int tile, hipStream_t stream);
int qmm_wo_ksplit_launch_f32_0(KsArgs& a, int tile, hipStream_t stream);
int qmm_wo_ksplit_launch_f32_1(KsArgs& a, int tile, hipStream_t stream);
