// Weight-only quantized matmul for a batch of rows (a decode batch of more than 16 sequences up to short prompts):
// per-channel int8 weights against bf16 / f16 rows, K split over the waves of a workgroup.
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
// What bounds it: 4 us that do not depend on K (launch, first loads, the sums through LDS), then about 75 KB per us
// and compute unit, x and weights together; at 64 x 48 per workgroup (100 x 6144 x 4096) the MFMAs alone would take
// 0.87 of the 1.05 us a step of 512 columns takes.  Measured with weights out of HBM / out of the Infinity Cache, us:
//   100 x 6144 x 4096      20.1 / 19.0  ->  14.3 / 12.1        32 x 4096 x 4096   9.9 / 9.1  ->  8.3 / 7.3
//   64 x 4096 x 4096       15.3 / 13.4  ->   9.5 /  8.3        32 x 1024 x 4096   7.9 / 7.5  ->  5.9 / 5.3
//   256 x 4096 x 4096      21.8 / 20.9  ->  15.1 / 12.9        48 x 3072 x 1536  11.0 / 9.6  ->  5.5 / 4.9
// Tried and not kept: streaming loads of the weights (no gain out of HBM, 0.5 - 1 us lost out of the cache); a deeper
// ring where ragged rows leave room for it; conversions placed by hand between the MFMAs (12.1 -> 12.8: the wave needs
// its weights a quarter of a step earlier); workgroups that start at different columns (within 3 % either way).
//
// This file is compiled per activation dtype and set of tiles (-DQMM_WO_XT=1|2 for bf16 | f16, -DQMM_KS_PART=0|1|2).
#include "qmm_common.h"
#include "qmm_frag.h"
#include "qmm_wo_gemm.h"

#if !defined(QMM_WO_XT) || !defined(QMM_KS_PART)
#error "compile with -DQMM_WO_XT=<XLA_AMD_DT_BF16|XLA_AMD_DT_F16 value> -DQMM_KS_PART=<0|1|2>"
#endif

namespace {

using namespace qmm_frag;

constexpr int kCopyWaves = 4;
constexpr int kLds = 160 * 1024;

// The launch's tiles: rows per tile (M spread evenly over the row tiles), row tiles, all tiles.
struct KsTiles {
  int rows, tiles_m, tiles;
  uint64_t tiles_m_magic;  // ceil(2^32 / tiles_m)
};

template <int MT, int NG, int KW, int CW> struct KsCfg {
  static constexpr int NW = KW * CW;             // computing waves
  static constexpr int BM = 16 * MT, BN = 16 * NG * CW;
  static constexpr int TILE = BM * 256;          // bytes of the x columns of one tile (128 columns, 2-byte x)
  static constexpr int SLOT = KW * TILE;
  static constexpr int PITCH = BN + 4;           // floats per row of the partial sums (4 more: rows start on other banks)
  static constexpr int kSums = KW * BM * (PITCH + 1) * 4;  // partial sums, and partial row sums of x
  static constexpr int kTail = 2 * BN * 4;       // scales and zero points as f32
  static constexpr int kFit = (kLds - kTail) / SLOT;
  static constexpr int R = kFit < 8 ? kFit : 8;  // slots of the ring
  static_assert(R >= 2, "the ring needs room to run ahead");
  static constexpr int lds_bytes(int steps) {
    const int ring = (steps < R ? steps : R) * SLOT;
    return kTail + (ring > kSums ? ring : kSums);
  }
  static_assert(kTail + kSums <= kLds, "the partial sums fit");
};

template <int XT, int MT, int NG, int KW, int CW, int P, bool HASZP, bool UNI>
__global__ void __launch_bounds__((KW * CW + kCopyWaves) * 64)
qmm_wo_ksplit_kernel(WoGemmArgs a, KsTiles t) {
  using Cfg = KsCfg<MT, NG, KW, CW>;
  constexpr int NW = Cfg::NW, BM = Cfg::BM, BN = Cfg::BN, TILE = Cfg::TILE, SLOT = Cfg::SLOT, R = Cfg::R, D = R - 1;
  constexpr int kThreads = (NW + kCopyWaves) * 64;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* const scl = (float*)smem;          // [BN] scales, [BN] zero points
  char* const ring = smem + Cfg::kTail;     // x slots; afterwards the partial sums
  float* const red = (float*)ring;          // [KW][BM][PITCH]
  float* const xsr = red + KW * BM * Cfg::PITCH;  // [KW][BM] partial row sums of x
  typedef __attribute__((address_space(3))) void* lds_ptr_t;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int M = a.M, N = a.N, K = a.K;
  // Workgroups are dealt round-robin to the 8 XCDs: each XCD gets a contiguous run of the tiles, row tiles fastest, so
  // that the row tiles of a column share its weights in that L2 (tile / tiles_m by multiply-shift: tile < 2^16).
  const int tile = ((int)blockIdx.x & 7) * (int)(gridDim.x >> 3) + ((int)blockIdx.x >> 3);
  if (tile >= t.tiles) return;
  const int col = (int)(((uint64_t)(uint32_t)tile * t.tiles_m_magic) >> 32);
  const int n0 = col * BN;
  const int m0 = (tile - col * t.tiles_m) * t.rows;
  const int rows = min(t.rows, M - m0);
  const int n_tiles = K / 128;
  const int steps = (n_tiles + KW - 1) / KW;
  const WoDts<XT, UNI> dts(a);

  f32x4 acc[NG][MT], xs[MT];
  uint32_t s_raw = 0, z_raw = 0;
  if (__builtin_expect(wave >= NW, 0)) {
    // ---- copying waves ----
    const int cw = wave - NW;
    const int quads = (rows + 3) >> 2;                         // an instruction copies four rows of 256 bytes
    const int nq = quads > cw ? (quads - cw + 3) >> 2 : 0;     // of this wave: cw, cw + 4, ...
    const char* const xb = (const char*)a.x + (size_t)m0 * K * 2;
    uint32_t x_off[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int row = min((cw + i * kCopyWaves) * 4 + (lane >> 4), rows - 1);
      x_off[i] = (uint32_t)row * ((uint32_t)K * 2u) + (uint32_t)(((lane & 15) ^ (row & 15)) * 16);
    }
    int issued = 0, slot = 0;
    auto issue = [&]() __attribute__((always_inline)) {
      char* const dst = ring + slot * SLOT;
#pragma unroll
      for (int k = 0; k < KW; ++k) {
        const char* const src = xb + (size_t)min(issued * KW + k, n_tiles - 1) * 256;
#pragma unroll
        for (int i = 0; i < MT; ++i)
          if (i < nq)
            __builtin_amdgcn_global_load_lds((const void*)(src + (size_t)x_off[i]), (lds_ptr_t)(dst + k * TILE + (cw + i * kCopyWaves) * 1024), 16, 0, 0);
      }
      ++issued;
      slot = slot + 1 == R ? 0 : slot + 1;
    };
    while (issued < min(D, steps)) issue();
    // the scales of the tile's channels: used at the very end
    if (cw * 64 + lane < BN) {
      const int n = min(n0 + cw * 64 + lane, N - 1);
      s_raw = qmm_load_raw(a.scale, n, dts.scale_dt);
      if constexpr (HASZP) z_raw = qmm_load_raw(a.zp, n, dts.zp_dt);
    }
    for (int n = 0; n < steps; ++n) {
      // the loads of the slots after n may be in flight (a wave's loads complete in order)
      const int ahead = issued - 1 - n;
      bool done = false;
      qmm_static_for<D>([&](auto dc) {
        qmm_static_for<MT + 1>([&](auto qc) {
          constexpr int c = (int)dc * KW * (int)qc;
          if (!done && ahead == (int)dc && nq == (int)qc) {
            qmm_wait_vmcnt<(c < 63 ? c : 63)>();
            done = true;
          }
        });
      });
      qmm_bare_barrier();  // slot n is there; the computing waves have read slot n - 1
      if (issued < steps) issue();
    }
    if (cw * 64 + lane < BN) {
      scl[cw * 64 + lane] = qmm_from_raw(s_raw, dts.scale_dt);
      if constexpr (HASZP) scl[BN + cw * 64 + lane] = qmm_from_raw(z_raw, dts.zp_dt);
    }
    qmm_bare_barrier();  // the computing waves have read the last slot
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
    qmm_static_for<MT>([&](auto mc) {
      xs[(int)mc] = f32x4{0, 0, 0, 0};
      qmm_static_for<NG>([&](auto gc) { acc[(int)gc][(int)mc] = f32x4{0, 0, 0, 0}; });
    });
    auto step = [&](int s, int slot, auto pc) __attribute__((always_inline)) {
      constexpr int p = pc;
      qmm_bare_barrier();
      const char* const xrow = ring + slot * SLOT + kw * TILE + r * 256;
      const bool live = s * KW + kw < n_tiles;  // (the last slot may hold fewer than KW tiles)
      i32x4 xq[2][MT];
      auto read = [&](auto jc) __attribute__((always_inline)) {
        constexpr int j = jc;
        qmm_static_for<MT>([&](auto mc) { xq[j & 1][(int)mc] = *(const i32x4*)(xrow + (int)mc * (16 * 256) + (((4 * g + j) ^ r) * 16)); });
      };
      read(qmm_const<0>{});
      qmm_static_for<4>([&](auto jc) {
        constexpr int j = jc;
        if constexpr (j < 3) read(qmm_const<j + 1>{});
        __builtin_amdgcn_sched_barrier(0);
        if (live) {
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
        if constexpr ((j & 1) == 1) request(s + P, pc, qmm_const<(j >> 1)>{});
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
        if (cw == 0 && g == 0) xsr[kw * BM + row] = xs[mt][0];
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
int launch(const WoGemmArgs& a, hipStream_t stream) {
  using Cfg = KsCfg<MT, NG, KW, CW>;
  KsTiles t;
  t.tiles_m = (a.M + Cfg::BM - 1) / Cfg::BM;
  t.rows = (a.M + t.tiles_m - 1) / t.tiles_m;
  t.tiles = t.tiles_m * ((a.N + Cfg::BN - 1) / Cfg::BN);
  t.tiles_m_magic = (((uint64_t)1 << 32) + t.tiles_m - 1) / t.tiles_m;
  const dim3 grid(8u * (unsigned)((t.tiles + 7) / 8)), block((Cfg::NW + kCopyWaves) * 64);
  const int steps = (a.K / 128 + KW - 1) / KW;
  auto go = [&](auto which) -> int {
    constexpr auto kern = decltype(which)::fn;
    static std::atomic<uint64_t> lds_set{0};
    const int rc = qmm_set_max_lds((const void*)kern, Cfg::lds_bytes(1 << 20), lds_set, "weight_only_gemm hipFuncSetAttribute");
    if (rc != XLA_AMD_QMM_OK) return rc;
    hipLaunchKernelGGL(kern, grid, block, Cfg::lds_bytes(steps), stream, a, t);
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
#else
#define QMM_KS_NAME QMM_KS_CAT(qmm_wo_ksplit_launch_f16_, QMM_KS_PART)
#endif
// tile: index into kKsTiles (qmm_wo_gemm.h)
int QMM_KS_NAME(const WoGemmArgs& a, int tile, hipStream_t stream) {
  switch (tile) {
#if QMM_KS_PART == 0
    case 0: return launch<QMM_WO_XT, 1, 1, 8, 1, 2>(a, stream);
    case 1: return launch<QMM_WO_XT, 1, 2, 8, 1, 2>(a, stream);
    case 2: return launch<QMM_WO_XT, 2, 1, 4, 2, 2>(a, stream);
    case 3: return launch<QMM_WO_XT, 2, 2, 4, 2, 1>(a, stream);
#elif QMM_KS_PART == 1
    case 4: return launch<QMM_WO_XT, 3, 2, 4, 1, 2>(a, stream);
    case 5: return launch<QMM_WO_XT, 3, 2, 4, 2, 1>(a, stream);
    case 6: return launch<QMM_WO_XT, 4, 2, 4, 2, 1>(a, stream);
#else
    case 7: return launch<QMM_WO_XT, 4, 3, 4, 2, 1>(a, stream);
    case 8: return launch<QMM_WO_XT, 4, 4, 4, 2, 1>(a, stream);
#endif
  }
  return qmm_fail(XLA_AMD_QMM_EINVAL, "weight_only_gemm: no such tile");
}
