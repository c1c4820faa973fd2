// Weight-only quantized matmul for a batch of rows against blockwise or int4 weights: K split over the waves of a
// workgroup.  The kernel of qmm_wo_ksplit.hip (its split of the work, x ring and operand paths) with the rounding points
// of the blockwise statements (qmm_wo_gemm_bw.hip): every wave takes whole quantization blocks - block b goes to the K
// group b % KW -, rounds each block's dot product, scales it and adds it up; what the waves add through LDS at the end
// are these sums (and those of the zero points' terms), which only need the final roundings.  Per-channel int4 weights
// (PERCH) have one block, whose raw sums are added.
//
// The tiled GEMM splits no K (100 rows against 4096 channels are 64 workgroups), and up to 64 rows the streaming kernel
// made a pass over the weight per 32.  Weights out of HBM / out of the Infinity Cache (geometric mean), us, int4 in blocks
// of 128 with zero points against 4096 x 4096: 32 rows 14.6 -> 8.9, 64 rows 28.4 -> 10.8, 128 rows 28.2 -> 14.4, 256 rows
// 28.5 -> 25; against 4096 x 14336 without: 64 rows 79 -> 27, 128 rows 82 -> 36.  Over 2500 drawn launches of 17 -
// 1000 rows, with the older kernels where they are estimated to be faster, 0.63 of the time (geometric mean).  What bounds it: fetching, as there, up to
// 32 rows; beyond, the vector instructions of a block's end (four to six per result and block).
//
// Arithmetic, one dtype (x's) throughout:
//   p_b = round(sum_block x w); out = round(sum_b scale_b p_b); zero point: out = round(out - round(sum_b round(sum_block x) zp_b)).
// int4 weights are expanded by an affine map (qmm_frag.h), its factor applied at the end.
//
// This file is compiled per activation dtype and bits (-DQMM_WO_XT=1|2 for bf16 | f16, -DQMM_KS_BITS=4|8).
#include "qmm_wo_bw.h"
#include "qmm_wo_ksplit.h"

#if !defined(QMM_WO_XT) || !defined(QMM_KS_BITS)
#error "compile with -DQMM_WO_XT=<XLA_AMD_DT_BF16|XLA_AMD_DT_F16 value> -DQMM_KS_BITS=<4|8>"
#endif

namespace {

template <int XT, int BITS, int MT, int NG, int KW, int CW, int P, bool HASZP, bool PERCH>
__global__ void __launch_bounds__((KW * CW + kCopyWaves) * 64)
qmm_wo_bw_gemm_kernel_ksplit(WoBwArgs a, KsTiles t) {
  using Cfg = KsCfg<XT, MT, NG, KW, CW, 0>;
  constexpr int NW = Cfg::NW, BM = Cfg::BM, BN = Cfg::BN, TILE = Cfg::TILE, SLOT = Cfg::SLOT, R = Cfg::R;
  constexpr int kThreads = (NW + kCopyWaves) * 64;
  constexpr bool NEEDXS = HASZP || BITS == 4;
  constexpr int BLK = BITS == 8 ? 2048 : 1024;  // bytes of one weight block (16 channels x 128 columns)
  constexpr int WL = BITS == 8 ? 2 : 1;         // 16-byte loads per lane and block
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* const ring = smem;                      // x slots; afterwards the partial sums
  float* const red = (float*)smem;              // [KW][BM][PITCH]
  float* const xsr = red + KW * BM * Cfg::PITCH;  // [KW][BM] partial row sums of x (PERCH)

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int M = a.M, N = a.N, K = a.K;
  int n0, m0, rows;
  if (!ks_tile_of(t, M, BN, n0, m0, rows)) return;
  const int n_tiles = K / 128;
  const int sub = PERCH ? 1 : a.C / 128;        // tiles per quantization block
  const int n_blocks = n_tiles / sub;           // (PERCH: every tile, what a wave adds up)
  const int steps = (n_blocks + KW - 1) / KW * sub;

  if (__builtin_expect(wave >= NW, 0)) {
    ks_copy_x<Cfg, KW>(
        a.x, K, m0, rows, steps, wave - NW, lane, ring,
        [&](int n, int k) {
          const int u = sub == 1 ? n : n / sub;
          return min((u * KW + k) * sub + (n - u * sub), n_tiles - 1);
        },
        []() {}, []() {});
  }
  f32x4 sacc[NG][MT], zacc[NG][MT], xs[MT];
  const int kw = wave / CW, cw = wave % CW;     // (of a computing wave)
  if (wave < NW) {
    const int groups = (N + 15) / 16;
    uint32_t w_lane[NG];  // this lane's 16 bytes of row set gi, from the tile's first group
    const uint8_t* const wp = a.w + (size_t)(n0 / 16) * n_tiles * BLK;
    qmm_static_for<NG>([&](auto gc) {
      const int grp = min(n0 / 16 + cw * NG + (int)gc, groups - 1) - n0 / 16;  // groups past N re-read the last one
      w_lane[(int)gc] = (uint32_t)grp * (uint32_t)n_tiles * (uint32_t)BLK + lane * 16u;
    });
    // the weights of this wave's tiles, and the scales and zero points of their blocks (four channels per lane), P tiles ahead
    i32x4 wreg[P][WL][NG];
    typedef int i32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));
    i32x2 sreg[P][NG], zreg[P][NG];
    int rq_u = 0, rq_t = 0;  // the next tile to request: tile rq_t of the wave's block rq_u
    auto request = [&](auto pc) __attribute__((always_inline)) {
      constexpr int p = pc;
      // (past the end: the last one again, no branch around the loads)
      const int blk = min(rq_u * KW + kw, n_blocks - 1);
      const int tile = min(blk * sub + rq_t, n_tiles - 1);
      const uint8_t* const src = wp + (size_t)tile * BLK;
      qmm_static_for<NG>([&](auto gc) {
        qmm_static_for<WL>([&](auto hc) { wreg[p][(int)hc][(int)gc] = *(const i32x4*)(src + (int)hc * 1024 + (size_t)w_lane[(int)gc]); });
        if constexpr (!PERCH) {
          const int n = min(n0 + (cw * NG + (int)gc) * 16 + 4 * g, N - 4);
          sreg[p][(int)gc] = *(const i32x2_a4*)((const uint16_t*)a.scale + (size_t)blk * N + n);
          if constexpr (HASZP) zreg[p][(int)gc] = *(const i32x2_a4*)((const uint16_t*)a.zp + (size_t)blk * N + n);
        }
      });
      if (++rq_t == sub) { rq_t = 0; ++rq_u; }
    };
    qmm_static_for<P>([&](auto pc) { request(pc); });
    __builtin_amdgcn_sched_barrier(0);
    f32x4 acc[NG][MT];
    qmm_static_for<MT>([&](auto mc) {
      xs[(int)mc] = f32x4{0, 0, 0, 0};
      qmm_static_for<NG>([&](auto gc) {
        acc[(int)gc][(int)mc] = f32x4{0, 0, 0, 0};
        sacc[(int)gc][(int)mc] = f32x4{0, 0, 0, 0};
        zacc[(int)gc][(int)mc] = f32x4{0, 0, 0, 0};
      });
    });
    int u = 0, ut = 0;  // the current tile: tile ut of the wave's block u
    auto step = [&](int slot, auto pc) __attribute__((always_inline)) {
      constexpr int p = pc;
      qmm_bare_barrier();
      const char* const xrow = ring + slot * SLOT + kw * TILE + r * 256;
      const bool live = u * KW + kw < n_blocks;  // (the last round of blocks may hold fewer than KW)
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
            i32x4 af;
            if constexpr (BITS == 8) {
              const i32x4 src = wreg[p][(j >> 1) % WL][gi];
              af = cvt_w8<XT>((uint32_t)src[(j & 1) * 2], (uint32_t)src[(j & 1) * 2 + 1]);
            } else {
              af = cvt_w4<XT>((uint32_t)wreg[p][0][gi][j]);
            }
            qmm_static_for<MT>([&](auto mc) { acc[gi][(int)mc] = mfma16<XT>(af, xq[j & 1][(int)mc], acc[gi][(int)mc]); });
          });
          if constexpr (NEEDXS) qmm_static_for<MT>([&](auto mc) { xs[(int)mc] = mfma16<XT>(ones_frag<XT>(), xq[j & 1][(int)mc], xs[(int)mc]); });
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (PERCH) {
        ++u;
      } else {
        if (++ut == sub) {
          if (live) {
            // the block's end: p = round(dot); sums += scale p; zero-point sums += round(sum x) zp
            qmm_static_for<NG>([&](auto gc) {
              constexpr int gi = gc;
              qmm_static_for<4>([&](auto vc) {
                constexpr int v = vc;
                const uint32_t sw = (uint32_t)sreg[p][gi][v >> 1];
                const float sc = qmm_from_raw((v & 1) ? (sw >> 16) : (sw & 0xffffu), XT);
                float zv = 0.f;
                if constexpr (HASZP) {
                  const uint32_t zw = (uint32_t)zreg[p][gi][v >> 1];
                  zv = qmm_from_raw((v & 1) ? (zw >> 16) : (zw & 0xffffu), XT);
                }
                qmm_static_for<MT>([&](auto mc) {
                  constexpr int mt = mc;
                  const float d = BITS == 4 ? fmaf(-kInt4Offset<XT>, xs[mt][0], acc[gi][mt][v]) : acc[gi][mt][v];
                  sacc[gi][mt][v] = fmaf(sc, qmm_round_dt(d, XT), sacc[gi][mt][v]);
                  if constexpr (HASZP) zacc[gi][mt][v] = fmaf(qmm_round_dt(xs[mt][0], XT), zv, zacc[gi][mt][v]);
                });
              });
              qmm_static_for<MT>([&](auto mc) { acc[gi][(int)mc] = f32x4{0, 0, 0, 0}; });
            });
            qmm_static_for<MT>([&](auto mc) { xs[(int)mc] = f32x4{0, 0, 0, 0}; });
          }
          ut = 0;
          ++u;
        }
      }
      request(pc);
      __builtin_amdgcn_sched_barrier(0);
    };
    int s = 0, slot = 0;
    for (; s + P <= steps; s += P)
      qmm_static_for<P>([&](auto pc) {
        step(slot, pc);
        slot = slot + 1 == R ? 0 : slot + 1;
      });
    qmm_static_for<P - 1>([&](auto pc) {
      if (s + (int)pc < steps) {
        step(slot, pc);
        slot = slot + 1 == R ? 0 : slot + 1;
      }
    });
    if constexpr (PERCH) qmm_static_for<MT>([&](auto mc) { qmm_static_for<NG>([&](auto gc) { sacc[(int)gc][(int)mc] = acc[(int)gc][(int)mc]; }); });
    qmm_bare_barrier();  // every wave has read the last slot: the ring takes the partial sums
  }

  // ---- the sums of the K groups, added in their order: a thread takes four channels of one row at a time ----
  constexpr int kQuads = BM * (BN / 4), kPer = (kQuads + kThreads - 1) / kThreads;
  auto put = [&](f32x4 (&v)[NG][MT]) __attribute__((always_inline)) {
    qmm_static_for<MT>([&](auto mc) {
      qmm_static_for<NG>([&](auto gc) {
        *(f32x4*)(red + ((size_t)kw * BM + 16 * (int)mc + r) * Cfg::PITCH + (cw * NG + (int)gc) * 16 + 4 * g) = v[(int)gc][(int)mc];
      });
    });
  };
  auto add = [&](int q) __attribute__((always_inline)) {
    const int row = q / (BN / 4), c = (q % (BN / 4)) * 4;
    f32x4 sum = *(const f32x4*)(red + (size_t)row * Cfg::PITCH + c);
#pragma unroll
    for (int k = 1; k < KW; ++k) sum += *(const f32x4*)(red + ((size_t)k * BM + row) * Cfg::PITCH + c);
    return sum;
  };
  if (wave < NW) {
    put(sacc);
    if constexpr (PERCH) {
      if (cw == 0 && g == 0) qmm_static_for<MT>([&](auto mc) { xsr[kw * BM + 16 * (int)mc + r] = xs[(int)mc][0]; });
    }
  }
  qmm_bare_barrier();
  constexpr float kFactor = BITS == 4 ? kInt4Factor<XT> : 1.0f;
  float o[kPer][4];
  qmm_static_for<kPer>([&](auto ic) {
    const int q = (int)ic * kThreads + (int)threadIdx.x;
    if (q < kQuads) {
      const f32x4 sum = add(q);
      if constexpr (PERCH) {
        const int row = q / (BN / 4), n = n0 + (q % (BN / 4)) * 4;
        float xsum = 0.f;
#pragma unroll
        for (int k = 0; k < KW; ++k) xsum += xsr[k * BM + row];
        qmm_static_for<4>([&](auto vc) {
          constexpr int v = vc;
          const int ch = min(n + v, N - 1);
          const float dot = kFactor * (BITS == 4 ? fmaf(-kInt4Offset<XT>, xsum, sum[v]) : sum[v]);
          float t = qmm_round_dt(qmm_load(a.scale, ch, XT) * qmm_round_dt(dot, XT), XT);
          if constexpr (HASZP) t = qmm_round_dt(t - qmm_round_dt(qmm_round_dt(xsum, XT) * qmm_load(a.zp, ch, XT), XT), XT);
          o[(int)ic][v] = t;
        });
      } else {
        qmm_static_for<4>([&](auto vc) { o[(int)ic][(int)vc] = qmm_round_dt(kFactor * sum[(int)vc], XT); });
      }
    }
  });
  if constexpr (HASZP && !PERCH) {
    qmm_bare_barrier();  // the sums have been read: the zero points' take their place
    if (wave < NW) put(zacc);
    qmm_bare_barrier();
    qmm_static_for<kPer>([&](auto ic) {
      const int q = (int)ic * kThreads + (int)threadIdx.x;
      if (q < kQuads) {
        const f32x4 z = add(q);
        qmm_static_for<4>([&](auto vc) { o[(int)ic][(int)vc] = qmm_round_dt(o[(int)ic][(int)vc] - qmm_round_dt(z[(int)vc], XT), XT); });
      }
    });
  }
  qmm_static_for<kPer>([&](auto ic) {
    const int q = (int)ic * kThreads + (int)threadIdx.x;
    const int row = q / (BN / 4), n = n0 + (q % (BN / 4)) * 4;
    if (q < kQuads && row < rows && n < N) wo_store4<true>(a.out, m0 + row, n, N, o[(int)ic], XT);  // N % 4 == 0
  });
}

// ZP: a tile for launches with a zero point too (96 more sums would not fit the registers of the largest one)
template <int XT, int BITS, int MT, int NG, int KW, int CW, int P, bool ZP = true>
int launch(const WoBwArgs& a, hipStream_t stream) {
  using Cfg = KsCfg<XT, MT, NG, KW, CW, 0>;
  const KsTiles t = ks_tiles(a.M, a.N, Cfg::BM, Cfg::BN);
  const dim3 grid(8u * (unsigned)t.per_xcd), block((Cfg::NW + kCopyWaves) * 64);
  const bool perch = a.C == a.K;
  const int sub = perch ? 1 : a.C / 128, blocks = a.K / 128 / sub;
  const int steps = (blocks + KW - 1) / KW * sub;
  auto go = [&](auto which) -> int {
    constexpr auto kern = decltype(which)::fn;
    static std::atomic<uint64_t> lds_set{0};
    const int rc = qmm_set_max_lds((const void*)kern, Cfg::lds_bytes(1 << 20), lds_set, "weight_only_gemm hipFuncSetAttribute");
    if (rc != XLA_AMD_QMM_OK) return rc;
    hipLaunchKernelGGL(kern, grid, block, Cfg::lds_bytes(steps), stream, a, t);
    return QMM_CHECK_LAUNCH("weight_only_gemm launch");
  };
  if constexpr (!ZP) {
    if (a.zp) return qmm_fail(XLA_AMD_QMM_EINVAL, "weight_only_gemm: no such tile with a zero point");
    if constexpr (BITS == 4) {
      if (perch) return go(qmm_kernel<qmm_wo_bw_gemm_kernel_ksplit<XT, BITS, MT, NG, KW, CW, P, false, true>>{});
    }
    return go(qmm_kernel<qmm_wo_bw_gemm_kernel_ksplit<XT, BITS, MT, NG, KW, CW, P, false, false>>{});
  } else {
    if constexpr (BITS == 4) {
      if (perch) return a.zp ? go(qmm_kernel<qmm_wo_bw_gemm_kernel_ksplit<XT, BITS, MT, NG, KW, CW, P, true, true>>{})
                             : go(qmm_kernel<qmm_wo_bw_gemm_kernel_ksplit<XT, BITS, MT, NG, KW, CW, P, false, true>>{});
    }
    return a.zp ? go(qmm_kernel<qmm_wo_bw_gemm_kernel_ksplit<XT, BITS, MT, NG, KW, CW, P, true, false>>{})
                : go(qmm_kernel<qmm_wo_bw_gemm_kernel_ksplit<XT, BITS, MT, NG, KW, CW, P, false, false>>{});
  }
}

}  // namespace

#define QMM_KS_CAT2(a, b) a##b
#define QMM_KS_CAT(a, b) QMM_KS_CAT2(a, b)
#if QMM_WO_XT == XLA_AMD_DT_BF16
#define QMM_KS_NAME QMM_KS_CAT(qmm_wo_ksplit_bw_launch_bf16_, QMM_KS_BITS)
#else
#define QMM_KS_NAME QMM_KS_CAT(qmm_wo_ksplit_bw_launch_f16_, QMM_KS_BITS)
#endif
// tile: index into kKsBwTiles (qmm_wo_bw.h)
int QMM_KS_NAME(const WoBwArgs& a, int tile, hipStream_t stream) {
  constexpr int B = QMM_KS_BITS;
  switch (tile) {
    case 0: return launch<QMM_WO_XT, B, 1, 1, 8, 1, 2>(a, stream);
    case 1: return launch<QMM_WO_XT, B, 1, 2, 8, 1, 2>(a, stream);
    case 2: return launch<QMM_WO_XT, B, 2, 1, 4, 2, 2>(a, stream);
    case 3: return launch<QMM_WO_XT, B, 3, 2, 4, 1, 2>(a, stream);
    case 4: return launch<QMM_WO_XT, B, 3, 2, 4, 2, 1>(a, stream);
    case 5: return launch<QMM_WO_XT, B, 4, 1, 4, 2, 2>(a, stream);
    case 6: return launch<QMM_WO_XT, B, 4, 2, 4, 2, 1, false>(a, stream);
  }
  return qmm_fail(XLA_AMD_QMM_EINVAL, "weight_only_gemm: no such tile");
}
