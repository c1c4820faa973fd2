// Weight-only quantized matmul for a batch of rows (a decode batch of more than 16 sequences up to short prompts) and for
// f32 rows: per-channel int8 weights, K split over the waves of a workgroup.
//
// Between the weight-streaming kernel (qmm_skinny.hip) and the tiled GEMM (qmm_wo_gemm.hip) lie the launches whose
// time is what every compute unit has to fetch: BM rows of x and BN channels of weights over all of K,
// (2 BM + BN) K bytes for a tile of BM x BN, with BM BN about M N / 256.  Tiles that small leave the computing waves
// little to share along rows or channels, so they share K: KW groups of CW waves take every KW th tile of 128 columns
// against the whole BM x BN tile (each x fragment read from LDS serves NG MFMAs, each converted weight fragment MT),
// and their sums are added through LDS at the end.  Nothing goes through memory but the operands and the results: the
// K slices over workgroups that such shapes took before wrote and read their partial sums (100 x 6144 x 4096: 12 MB
// in five slices, and a second kernel), and the streaming kernel stopped for every chunk of two x tiles.
//
// Weights come from the tiled copy straight into registers, as in qmm_wo_gemm.hip (MFMA row sets of 16 consecutive
// channels whatever the group width G), P tiles ahead.  x goes through LDS in a ring of R slots of KW tiles, filled
// R - 1 slots ahead by four copying waves (global -> LDS without registers; only live rows are copied); the workgroup
// meets once per slot.  MFMA mapping and arithmetic are those of qmm_wo_gemm.hip.
//
// What bounds it: 4 us that do not depend on K (launch, first loads, the sums through LDS), then waiting: 60 - 75 KB per us
// and compute unit arrive, x and weights together, where the copies of an LDS-tiled kernel reach 110 - 130 out of L2.  By
// counters the waves wait for data or at the barrier of each slot in 61 % of their cycles (64 x 4096 x 4096, 32 x 32 tiles on
// 256 compute units; the MFMAs are busy 11 % of the time, LDS conflicts cost 12 %), in 51 % for 100 x 6144 x 4096 with a zero
// point (64 x 64 tiles, 192 workgroups; MFMAs 39 %, a third of them the row sums of x, which both waves along the channels
// make).  Measured with weights out of HBM / out of the Infinity Cache, us:
//   100 x 6144 x 4096      20.1 / 19.0  ->  14.0 / 12.1        32 x 4096 x 4096   9.9 / 9.1  ->  8.3 / 7.3
//   64 x 4096 x 4096       15.3 / 13.4  ->   9.5 /  8.3        32 x 1024 x 4096   7.9 / 7.5  ->  5.9 / 5.3
//   256 x 4096 x 4096      21.8 / 20.9  ->  15.1 / 12.9        48 x 3072 x 1536  11.0 / 9.6  ->  5.5 / 4.9
// Tried and not kept: streaming loads of the weights (no gain out of HBM, 0.5 - 1 us lost out of the cache); a deeper
// ring where ragged rows leave room for it; conversions placed by hand between the MFMAs (12.1 -> 12.8: the wave needs
// its weights a quarter of a step earlier); workgroups that start at different columns (within 3 % either way).
//
// f32 rows (below 128, and more where the launch has few tiles) run the same kernel on 16x16x4 f32
// MFMAs, one column per lane and instruction: true f32 products, an eighth of the bf16 rate, so the matrix cores bound
// all but the smallest launches (64 x 4096 x 4096: 22 us, 14 of them MFMAs).  The streaming kernel before it made a pass
// over the weight per 16 rows and split K over two waves at most, 512 columns each: 8 x 1024 x 1024 6.6 -> 4.6 us, 32 x
// 4096 x 4096 25.6 -> 14.4, 100 x 1024 x 1024 43 -> 6.5; over 300 drawn launches of 1 - 127 rows 0.53 of the time (geometric
// mean, as below).  f32 MFMAs are busy 66 % of the cycles at 64 x 4096 x 4096.
//
// Over 2500 drawn launches of 17 - 1000 rows of 2-byte x (N 512 - 14336, K 1024 - 14336, weights out of HBM), with the older
// kernels where they are estimated to be faster, 0.61 of the time of the kernels before.
//
// This file is compiled per activation dtype and set of tiles (-DQMM_WO_XT=0|1|2 for f32 | bf16 | f16, -DQMM_KS_PART=0|1|2).
#include "qmm_wo_ksplit.h"

#if !defined(QMM_WO_XT) || !defined(QMM_KS_PART)
#error "compile with -DQMM_WO_XT=<XLA_AMD_DT_F32|XLA_AMD_DT_BF16|XLA_AMD_DT_F16 value> -DQMM_KS_PART=<0|1|2>"
#endif

namespace {

// scales and zero points of the tile as f32
template <int NG, int CW> constexpr int ks_tail() { return 2 * 16 * NG * CW * 4; }

template <int XT, int MT, int NG, int KW, int CW, int P, bool HASZP, bool UNI>
__global__ void __launch_bounds__((KW * CW + kCopyWaves) * 64)
qmm_wo_ksplit_kernel(KsArgs a) {
  using Cfg = KsCfg<XT, MT, NG, KW, CW, ks_tail<NG, CW>()>;
  constexpr bool kF32 = XT == XLA_AMD_DT_F32;
  constexpr int NW = Cfg::NW, BM = Cfg::BM, BN = Cfg::BN, TILE = Cfg::TILE, SLOT = Cfg::SLOT, R = Cfg::R;
  constexpr int kThreads = (NW + kCopyWaves) * 64;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* const scl = (float*)smem;             // [BN] scales, [BN] zero points
  char* const ring = smem + ks_tail<NG, CW>(); // x slots; afterwards the partial sums
  float* const red = (float*)ring;             // [KW][BM][PITCH]
  float* const xsr = red + KW * BM * Cfg::PITCH;  // [KW][BM] partial row sums of x

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int M = a.M, N = a.N, K = a.K;
  int n0, m0, rows;
  if (!ks_tile_of(a.t, M, BN, n0, m0, rows)) return;
  const int n_tiles = K / 128;
  const int steps = (n_tiles + KW - 1) / KW;
  const WoDts<XT, UNI> dts(a);

  if (__builtin_expect(wave >= NW, 0)) {
    // ---- copying waves: x, and the scales of the tile's channels, which are used at the very end ----
    const int cw = wave - NW;
    uint32_t s_raw = 0, z_raw = 0;
    ks_copy_x<Cfg, KW>(
        a.x, K, m0, rows, steps, cw, lane, ring, [&](int n, int k) { return min(n * KW + k, n_tiles - 1); },
        [&]() {
          if (cw * 64 + lane < BN) {
            const int n = min(n0 + cw * 64 + lane, N - 1);
            s_raw = qmm_load_raw(a.scale, n, dts.scale_dt);
            if constexpr (HASZP) z_raw = qmm_load_raw(a.zp, n, dts.zp_dt);
          }
        },
        [&]() {
          if (cw * 64 + lane < BN) {
            scl[cw * 64 + lane] = qmm_from_raw(s_raw, dts.scale_dt);
            if constexpr (HASZP) scl[BN + cw * 64 + lane] = qmm_from_raw(z_raw, dts.zp_dt);
          }
        });
  } else {
    // ---- computing waves: wave (kw, cw) multiplies the tiles kw, kw + KW, ... against its NG row sets of 16 channels ----
    const int kw = wave / CW, cw = wave % CW;
    const int G = a.G, n_blk = K / 128;
    const int blk_bytes = G * 128, half_bytes = G * 64;
    // (divisions by G as in qmm_wo_gemm.hip: t < 272)
    const uint32_t g_magic = (65536u + (uint32_t)G - 1u) / (uint32_t)G;
    const int p0 = n0 / G, a0 = n0 - p0 * G;
    const uint8_t* const wp = a.w + (size_t)p0 * n_blk * blk_bytes;
    uint32_t w_lane[NG];
    qmm_static_for<NG>([&](auto gc) {
      constexpr int gi = gc;
      const uint32_t t = (uint32_t)(a0 + min((cw * NG + gi) * 16 + r, N - 1 - n0));
      const uint32_t pd = (t * g_magic) >> 16, row = t - pd * (uint32_t)G;
      w_lane[gi] = pd * ((uint32_t)n_blk * (uint32_t)blk_bytes) + ((uint32_t)(g * G) + row) * 16u;
    });
    i32x4 wreg[P][2][NG];
    // half h of this wave's tile s (a tile past the end is the last one again: no branch around the loads)
    auto request = [&](int s, auto pc, auto hc) __attribute__((always_inline)) {
      constexpr int p = pc, h = hc;
      const uint8_t* const half = wp + (size_t)min(s * KW + kw, n_tiles - 1) * blk_bytes + h * half_bytes;
      qmm_static_for<NG>([&](auto gc) {
        wreg[p][h][(int)gc] = *(const i32x4*)(half + (size_t)w_lane[(int)gc]);
      });
    };
    qmm_static_for<P>([&](auto pc) {
      request((int)pc, pc, qmm_const<0>{});
      request((int)pc, pc, qmm_const<1>{});
    });
    __builtin_amdgcn_sched_barrier(0);
    f32x4 acc[NG][MT], xs[MT];
    qmm_static_for<MT>([&](auto mc) {
      xs[(int)mc] = f32x4{0, 0, 0, 0};
      qmm_static_for<NG>([&](auto gc) { acc[(int)gc][(int)mc] = f32x4{0, 0, 0, 0}; });
    });
    auto step = [&](int s, int slot, auto pc) __attribute__((always_inline)) {
      constexpr int p = pc;
      qmm_bare_barrier();
      const char* const xrow = ring + slot * SLOT + kw * TILE + r * Cfg::ROW;
      const bool live = s * KW + kw < n_tiles;  // (the last slot may hold fewer than KW tiles)
      constexpr int J = Cfg::ROW / 64;  // 16-byte pieces of a row of the tile per lane
      i32x4 xq[2][MT];
      auto read = [&](auto jc) __attribute__((always_inline)) {
        constexpr int j = jc;
        qmm_static_for<MT>([&](auto mc) { xq[j & 1][(int)mc] = *(const i32x4*)(xrow + (int)mc * (16 * Cfg::ROW) + (((J * g + j) ^ r) * 16)); });
      };
      read(qmm_const<0>{});
      qmm_static_for<J>([&](auto jc) {
        constexpr int j = jc;
        if constexpr (j + 1 < J) read(qmm_const<j + 1>{});
        __builtin_amdgcn_sched_barrier(0);
        if (live) {
          if constexpr (kF32) {
            // columns 32 g + 4 j .. + 3, one per instruction (true f32 products); their sum by vector instructions: an
            // MFMA against ones takes as long as one against weights
            qmm_static_for<4>([&](auto ec) {
              constexpr int e = ec;
              qmm_static_for<NG>([&](auto gc) {
                const float wf = (float)(int8_t)((uint32_t)wreg[p][j >> 2][(int)gc][j & 3] >> (8 * e));
                qmm_static_for<MT>([&](auto mc) {
                  acc[(int)gc][(int)mc] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf, __builtin_bit_cast(f32x4, xq[j & 1][(int)mc])[e], acc[(int)gc][(int)mc], 0, 0, 0);
                });
              });
              if constexpr (HASZP) qmm_static_for<MT>([&](auto mc) { xs[(int)mc][e] += __builtin_bit_cast(f32x4, xq[j & 1][(int)mc])[e]; });
            });
          } else {
            qmm_static_for<NG>([&](auto gc) {
              constexpr int gi = gc;
              const i32x4 src = wreg[p][j >> 1][gi];
              const i32x4 af = cvt_w8<XT>((uint32_t)src[(j & 1) * 2], (uint32_t)src[(j & 1) * 2 + 1]);
              qmm_static_for<MT>([&](auto mc) { acc[gi][(int)mc] = mfma16<XT>(af, xq[j & 1][(int)mc], acc[gi][(int)mc]); });
            });
            if constexpr (HASZP) {
              qmm_static_for<MT>([&](auto mc) { xs[(int)mc] = mfma16<XT>(ones_frag<XT>(), xq[j & 1][(int)mc], xs[(int)mc]); });
            }
          }
        }
        if constexpr (j % (J / 2) == J / 2 - 1) request(s + P, pc, qmm_const<j / (J / 2)>{});
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    int s = 0, slot = 0;
    for (; s + P <= steps; s += P)
      qmm_static_for<P>([&](auto pc) {
        step(s + (int)pc, slot, pc);
        slot = slot + 1 == R ? 0 : slot + 1;
      });
    qmm_static_for<P - 1>([&](auto pc) {
      if (s + (int)pc < steps) {
        step(s + (int)pc, slot, pc);
        slot = slot + 1 == R ? 0 : slot + 1;
      }
    });
    qmm_bare_barrier();  // every wave has read the last slot: the ring takes the partial sums
    qmm_static_for<MT>([&](auto mc) {
      constexpr int mt = mc;
      const int row = 16 * mt + r;
      qmm_static_for<NG>([&](auto gc) {
        constexpr int gi = gc;
        *(f32x4*)(red + ((size_t)kw * BM + row) * Cfg::PITCH + (cw * NG + gi) * 16 + 4 * g) = acc[gi][mt];
      });
      if constexpr (HASZP) {
        float sum = xs[mt][0];
        if constexpr (kF32) {  // four of the lane's columns each, and a quarter of the row per lane
          sum = (xs[mt][0] + xs[mt][1]) + (xs[mt][2] + xs[mt][3]);
          sum += __shfl_xor(sum, 16);
          sum += __shfl_xor(sum, 32);
        }
        if (cw == 0 && g == 0) xsr[kw * BM + row] = sum;
      }
    });
  }
  qmm_bare_barrier();  // the partial sums and the scales are in LDS

  // ---- results: a thread adds the KW sums of four channels of one row, in wave order ----
  for (int q = threadIdx.x; q < BM * (BN / 4); q += kThreads) {
    const int row = q / (BN / 4), c = (q % (BN / 4)) * 4;
    const int m = m0 + row, n = n0 + c;
    if (row >= rows || n >= N) continue;
    f32x4 dot = *(const f32x4*)(red + (size_t)row * Cfg::PITCH + c);
#pragma unroll
    for (int k = 1; k < KW; ++k) dot += *(const f32x4*)(red + ((size_t)k * BM + row) * Cfg::PITCH + c);
    float xsum = 0.f;
    if constexpr (HASZP) {
#pragma unroll
      for (int k = 0; k < KW; ++k) xsum += xsr[k * BM + row];
    }
    float o[4];
    wo_finish4_f(dts, scl + c, scl + BN + c, HASZP, dot, xsum, dts.x_dt, o);
    if ((N & 3) == 0) wo_store4<true>(a.out, m, n, N, o, dts.store_dt);
    else wo_store4<false>(a.out, m, n, N, o, dts.store_dt);
  }
}

template <int XT, int MT, int NG, int KW, int CW, int P>
int launch(KsArgs& a, hipStream_t stream) {
  using Cfg = KsCfg<XT, MT, NG, KW, CW, ks_tail<NG, CW>()>;
  a.t = ks_tiles(a.M, a.N, Cfg::BM, Cfg::BN);
  const dim3 grid(8u * (unsigned)a.t.per_xcd), block((Cfg::NW + kCopyWaves) * 64);
  const int steps = (a.K / 128 + KW - 1) / KW;
  auto go = [&](auto which) -> int {
    constexpr auto kern = decltype(which)::fn;
    static std::atomic<uint64_t> lds_set{0};
    const int rc = qmm_set_max_lds((const void*)kern, Cfg::lds_bytes(1 << 20), lds_set, "weight_only_gemm hipFuncSetAttribute");
    if (rc != XLA_AMD_QMM_OK) return rc;
    hipLaunchKernelGGL(kern, grid, block, Cfg::lds_bytes(steps), stream, a);
    return QMM_CHECK_LAUNCH("weight_only_gemm launch");
  };
  const bool uni = a.scale_dt == XT && a.zp_dt == XT && a.dot_dt == XT && a.out_dt == XT && a.store_dt == XT;
  if (uni) return a.zp ? go(qmm_kernel<qmm_wo_ksplit_kernel<XT, MT, NG, KW, CW, P, true, true>>{})
                       : go(qmm_kernel<qmm_wo_ksplit_kernel<XT, MT, NG, KW, CW, P, false, true>>{});
  return a.zp ? go(qmm_kernel<qmm_wo_ksplit_kernel<XT, MT, NG, KW, CW, P, true, false>>{})
              : go(qmm_kernel<qmm_wo_ksplit_kernel<XT, MT, NG, KW, CW, P, false, false>>{});
}

}  // namespace

#define QMM_KS_CAT2(a, b) a##b
#define QMM_KS_CAT(a, b) QMM_KS_CAT2(a, b)
#if QMM_WO_XT == XLA_AMD_DT_BF16
#define QMM_KS_NAME QMM_KS_CAT(qmm_wo_ksplit_launch_bf16_, QMM_KS_PART)
#elif QMM_WO_XT == XLA_AMD_DT_F16
#define QMM_KS_NAME QMM_KS_CAT(qmm_wo_ksplit_launch_f16_, QMM_KS_PART)
#else
#define QMM_KS_NAME QMM_KS_CAT(qmm_wo_ksplit_launch_f32_, QMM_KS_PART)
#endif
// tile: index into kKsTiles, or kKsTilesF32 (qmm_wo_gemm.h)
int QMM_KS_NAME(KsArgs& a, int tile, hipStream_t stream) {
  switch (tile) {
#if QMM_WO_XT == XLA_AMD_DT_F32
#if QMM_KS_PART == 0
    case 0: return launch<QMM_WO_XT, 1, 1, 8, 1, 2>(a, stream);
    case 1: return launch<QMM_WO_XT, 1, 2, 8, 1, 2>(a, stream);
    case 2: return launch<QMM_WO_XT, 1, 4, 8, 1, 1>(a, stream);
#elif QMM_KS_PART == 1
    case 3: return launch<QMM_WO_XT, 1, 1, 4, 1, 2>(a, stream);
    case 4: return launch<QMM_WO_XT, 2, 1, 4, 2, 2>(a, stream);
    case 5: return launch<QMM_WO_XT, 2, 2, 4, 2, 1>(a, stream);
#endif
#elif QMM_KS_PART == 0
    case 0: return launch<QMM_WO_XT, 1, 1, 8, 1, 2>(a, stream);
    case 1: return launch<QMM_WO_XT, 1, 2, 8, 1, 2>(a, stream);
    case 2: return launch<QMM_WO_XT, 2, 1, 4, 2, 2>(a, stream);
    case 3: return launch<QMM_WO_XT, 2, 2, 4, 2, 1>(a, stream);
#elif QMM_KS_PART == 1
    case 4: return launch<QMM_WO_XT, 3, 2, 4, 1, 2>(a, stream);
    case 5: return launch<QMM_WO_XT, 3, 2, 4, 2, 1>(a, stream);
    case 6: return launch<QMM_WO_XT, 4, 2, 4, 2, 1>(a, stream);
#elif QMM_KS_PART == 2
    case 7: return launch<QMM_WO_XT, 4, 3, 4, 2, 1>(a, stream);
    case 8: return launch<QMM_WO_XT, 4, 4, 4, 2, 1>(a, stream);
#endif
  }
  return qmm_fail(XLA_AMD_QMM_EINVAL, "weight_only_gemm: no such tile");
}
