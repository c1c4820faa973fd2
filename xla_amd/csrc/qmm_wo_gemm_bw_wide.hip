// Weight-only quantized matmul for many rows of x with blockwise or int4 weights, for launches with many tiles: the
// tiled MFMA GEMM of qmm_wo_gemm_bw.hip (its operands, arithmetic and rounding points) over tiles of 64 rows x 256
// channels, with eight computing waves instead of four.
//
// What bounds it: instruction issue.  A step of a wave (64 rows x 32 channels x 128 columns) is 32 MFMAs, and beside
// them the expansion of the weights (64 instructions for int4) and the block's rounding sequence (72 in
// bf16, see wo_bw_round2; 88 in f16).  On a SIMD an
// MFMA takes about 13 cycles of issue and every other vector instruction 4, whichever of its waves they come from, so
// what counts is how few instructions a step has:
//  * the sums of x per step come from the copying waves, once per row (four MFMAs against ones for their 16 rows)
//    instead of once per row and computing wave, and reach the computing waves as the MFMAs' initial accumulators
//    (-kInt4Offset sum x, four times side by side: a lane reads its accumulator quad), so that undoing the affine map of
//    int4 weights (qmm_frag.h) costs no vector instruction;
//  * the zero points' term is a matrix product over the blocks: the copying waves leave round_x(sum x) of 16 blocks
//    in LDS, next to the zero points of the 16 blocks, and the computing waves add them with one MFMA per result tile.
// The second wave per SIMD covers the waits of the first, and twice the channels per workgroup halve the copies of x.
// 2048 rows against 4096 x 4096, bf16, blocks of 128, per launch in a graph (this kernel / the 64 x 128 tile, one box; from
// box to box 75 - 86 / 108 - 121): int4 with zero point 81 / 114 us, without 77 / 105, int8 84 / 97; per-channel int4
// 69 / 90.  Everything but the MFMAs, expansion and rounding switched off it takes 65 us.
#include "qmm_common.h"
#include "qmm_frag.h"
#include "qmm_wo_bw.h"

#ifndef QMM_WO_BW_XT
#error "compile with -DQMM_WO_BW_XT=<XLA_AMD_DT_BF16|XLA_AMD_DT_F16 value>"
#endif

namespace {

using namespace qmm_frag;

constexpr int kComputeWaves = 8;
constexpr int kCopyWaves = 4;
constexpr int NG = 2;                    // channel groups of 16 per computing wave
constexpr int BM = 64;                   // rows of x per workgroup
constexpr int X_TILE = BM * 256;         // bytes of the x columns of one step (128 columns, 2-byte x)
constexpr int CS = 4;                    // steps per chunk slot
constexpr int kZBlocks = 16;             // quantization blocks per zero-point product
static_assert(BM == 16 * kCopyWaves, "a copying wave copies and sums the 16 rows of one MFMA tile");

constexpr int MT = BM / 16;              // 16-row tiles: every computing wave owns all rows of its channels
constexpr int BN = 16 * NG * kComputeWaves;  // 256 channels per workgroup
constexpr int kEntry = BN * 2;           // one entry: the workgroup's channels, 2-byte values
// LDS: scales of every resident step; -kInt4Offset sum x of every resident step and row, four times; zero points and rounded
// sums of x of two groups of 16 blocks; x
constexpr int kXsq = 2 * CS * kEntry;
constexpr int kZent = kXsq + 2 * CS * BM * 16;
constexpr int kZx = kZent + 2 * kZBlocks * kEntry;
constexpr int kX = kZx + 2 * kZBlocks * BM * 2;
constexpr int kLdsBytes = kX + 2 * CS * X_TILE;
static_assert(kLdsBytes <= 160 * 1024, "LDS of a compute unit");

struct BwItem {
  int m0, n0, rows;
};

// BLK1: quantization blocks of 128 columns, one per step.  With a zero point there is no other form.
template <int XT, int BITS, bool HASZP, bool BLK1>
__global__ void __launch_bounds__((kComputeWaves + kCopyWaves) * 64)
qmm_wo_bw_wide_kernel(WoBwArgs a) {
  static_assert(BLK1 || !HASZP, "zero points: one block per step");
  constexpr bool NEEDXS = HASZP || BITS == 4;        // sums of x: zero point, int4 affine map
  constexpr int BLK = BITS == 8 ? 2048 : 1024;       // bytes of one weight block (16 channels x 128 columns)
  constexpr int WL = BITS == 8 ? 2 : 1;              // 16-byte loads per lane and block
  extern __shared__ __attribute__((aligned(16))) char smem[];
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  char* const xsm = smem + kX;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int M = a.M, N = a.N, K = a.K;
  const int steps = K / 128;
  const int n_chunks = (steps + CS - 1) / CS;
  const int sub = BLK1 ? 1 : a.C / 128;              // steps per quantization block
  const int z_groups = (steps / sub + kZBlocks - 1) / kZBlocks;  // zero-point products per item
  const int tiles_n = (N + BN - 1) / BN;
  const int n_items = tiles_n * ((M + BM - 1) / BM);
  // item -> (row tile, column tile), column tiles fastest: workgroups that run together share x rows
  auto item_of = [&](int it) __attribute__((always_inline)) {
    BwItem w;
    w.m0 = (it / tiles_n) * BM;
    w.n0 = (it % tiles_n) * BN;
    w.rows = min(BM, M - w.m0);
    return w;
  };

  if (__builtin_expect(wave >= kComputeWaves, 0)) {
    // ---- copying waves: chunk after chunk of x (and its scales, zero points and sums) into the two slots in turn.
    // Wave cw copies the rows 16 cw .. 16 cw + 15 and sums what it has copied itself.
    const int cw = wave - kComputeWaves;
    int blk = 0;  // current step of the item, which with a zero point is a quantization block
    // one entry (the workgroup's channels of row `at` of a [K/C, N] tensor): 4 bytes (two channels) per lane
    auto copy_entry = [&](const void* from, int at, int n0, char* to) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < BN / 128; ++i) {
        const int ch = min(n0 + 128 * i + 2 * lane, N - 2);  // channels past N: any valid address (never used)
        __builtin_amdgcn_global_load_lds((const void*)((const char*)from + ((size_t)at * N + ch) * 2),
                                         (lds_ptr_t)(to + 256 * i), 4, 0, 0);
      }
    };
    auto chunk_load = [&](const BwItem& w, int c, int slot_i, int zg0) __attribute__((always_inline)) {
      const int s0 = c * CS;
      const int nst = min(CS, steps - s0);
      // step s0 + cw: its scales, and zero points
      static_assert(CS == kCopyWaves, "one step's entries per copying wave");
      if (cw < nst) {
        const int at = (s0 + cw) / sub;
        copy_entry(a.scale, at, w.n0, smem + (slot_i * CS + cw) * kEntry);
        if constexpr (HASZP)
          copy_entry(a.zp, at, w.n0, smem + kZent + (((zg0 + at / kZBlocks) & 1) * kZBlocks + at % kZBlocks) * kEntry);
      }
      char* const slot = xsm + slot_i * (CS * X_TILE);
      const char* const xb = (const char*)a.x + (size_t)w.m0 * K * 2;
      // a row of one step is 256 bytes: an instruction copies four consecutive rows
      // (lane l: row l/16 of the four, chunk l%16), swizzled on the source side
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r4 = 16 * cw + 4 * i;
        if (r4 < w.rows) {
          const int row = min(r4 + (lane >> 4), w.rows - 1);  // rows past the end repeat the last one
          const int chunk = (lane & 15) ^ (row & 15);
          const char* src = xb + (size_t)row * ((size_t)K * 2) + (size_t)s0 * 256 + chunk * 16;
          char* dst = slot + r4 * 256;
          for (int t = 0; t < nst; ++t)
            __builtin_amdgcn_global_load_lds((const void*)(src + t * 256), (lds_ptr_t)(dst + t * X_TILE), 16, 0, 0);
        }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if constexpr (NEEDXS) {
        if (c == 0) blk = 0;
        for (int t = 0; t < nst; ++t) {
          const char* xrow = slot + t * X_TILE + (16 * cw + r) * 256;
          f32x4 xs = {0, 0, 0, 0};
          qmm_static_for<4>([&](auto jc) {
            xs = mfma16<XT>(ones_frag<XT>(), *(const i32x4*)(xrow + (((4 * g + (int)jc) ^ r) * 16)), xs);
          });
          const float s = xs[0];  // (the same in every lane of a row)
          if constexpr (BITS == 4) {
            const float q = -kInt4Offset<XT> * s;
            if (g == 0) *(f32x4*)(smem + kXsq + ((slot_i * CS + t) * BM + 16 * cw + r) * 16) = f32x4{q, q, q, q};
          }
          if constexpr (HASZP) {
            const uint16_t v = XT == XLA_AMD_DT_BF16 ? qmm_f32_to_bf16(s) : qmm_f32_to_f16(s);
            if (g == 0)
              *(uint16_t*)(smem + kZx + ((((zg0 + blk / kZBlocks) & 1) * BM + 16 * cw + r) * kZBlocks + blk % kZBlocks) * 2) = v;
            ++blk;
          }
        }
      }
    };
    int it = blockIdx.x;
    BwItem cur = item_of(it);
    int c = 0, ring = 0, zg0 = 0;  // ring: chunks since the kernel began; chunk `ring` lives in slot ring % 2
    chunk_load(cur, 0, 0, 0);
    for (;;) {
      qmm_bare_barrier();  // chunk `ring` is there, chunk ring - 1 has been read
      ++c; ++ring;
      if (c == n_chunks) {
        it += gridDim.x;
        if (it >= n_items) break;
        cur = item_of(it);
        c = 0;
        zg0 += z_groups;
      }
      chunk_load(cur, c, ring & 1, zg0);
    }
    return;
  }

  // ---- computing waves ----
  // wave w owns the channel groups n0/16 + w*NG .. + NG-1
  const int n_blk = K / 128;  // blocks per channel group in the tiled weight
  const int groups = (N + 15) / 16;
  const uint8_t* wp[NG];
  auto set_weights = [&](const BwItem& w) __attribute__((always_inline)) {
    qmm_static_for<NG>([&](auto gc) {
      constexpr int gi = gc;
      const int grp = min(w.n0 / 16 + wave * NG + gi, groups - 1);  // groups past N re-read the last one
      wp[gi] = a.w + (size_t)grp * n_blk * BLK;
    });
  };
  // the weights of a step are requested a whole step ahead: step s of an item in slot s % 2
  i32x4 wreg[2][NG][WL];
  uint32_t w_off = lane * 16;
  auto load_w = [&](int blk, auto pc) __attribute__((always_inline)) {
    constexpr int P = pc;
    asm volatile("" : "+v"(w_off));  // (scalar base + 32-bit lane offset, not a 64-bit address per group in registers)
    qmm_static_for<NG>([&](auto gc) {
      constexpr int gi = gc;
      qmm_static_for<WL>([&](auto hc) {
        constexpr int h = hc;
        // (an ordinary load, not a streaming one: the other row tiles read the same block out of L2)
        wreg[P][gi][h] = *(const i32x4*)(wp[gi] + (size_t)blk * BLK + h * 1024 + (size_t)w_off);
      });
    });
  };

  f32x4 acc[NG][MT], sacc[NG][MT], zacc[NG][MT];
  // this lane's LDS addresses: its first 16 bytes of the first row tile (those of j lie at this address ^ 16 j), its
  // row's sum of x, its channels' scales
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
  const uint32_t x_at = lds0 + (uint32_t)(kX + r * 256 + ((4 * g) ^ r) * 16);
  const uint32_t xsq_at = lds0 + (uint32_t)(kXsq + r * 16);
  const uint32_t ent_at = lds0 + (uint32_t)((wave * NG * 16 + 4 * g) * 2);
  typedef __attribute__((address_space(3))) const i32x4* lds_i4_t;
  typedef __attribute__((address_space(3))) const f32x4* lds_f4_t;
  typedef __attribute__((address_space(3))) const i32x2* lds_i2_t;

  // End of quantization block: p = round(acc) and out_acc += scale p, with the scales of step k of LDS slot `slot`.
  auto round_block = [&](int slot, auto kc) __attribute__((always_inline)) {
    const uint32_t ent = ent_at + (uint32_t)slot * (CS * kEntry);
    qmm_static_for<NG>([&](auto gc) {
      constexpr int gi = gc;
      const i32x2 sraw = *(lds_i2_t)(uintptr_t)(ent + (int)kc * kEntry + gi * 32);
      qmm_static_for<4>([&](auto vc) {
        constexpr int v = vc;
        const uint32_t sw = (uint32_t)sraw[v >> 1];
        const float sc = qmm_from_raw((v & 1) ? (sw >> 16) : (sw & 0xffffu), XT);
        qmm_static_for<MT / 2>([&](auto mc) {
          constexpr int mt = 2 * (int)mc;
          const float d0 = acc[gi][mt][v], d1 = acc[gi][mt + 1][v];
          float p0, p1;
          wo_bw_round2<XT>(d0, d1, p0, p1);
          sacc[gi][mt][v] = fmaf(sc, p0, sacc[gi][mt][v]);
          sacc[gi][mt + 1][v] = fmaf(sc, p1, sacc[gi][mt + 1][v]);
        });
      });
      // (here: the compiler would sink it behind the zero points' product, with the accumulators live meanwhile)
      if constexpr (HASZP) qmm_static_for<MT>([&](auto mc) { f32x4 t = sacc[gi][(int)mc]; asm volatile("" : "+v"(t)); sacc[gi][(int)mc] = t; });
    });
  };
  // z_acc += round(sum x) zp over the first `count` blocks of LDS group `zg`: one MFMA per result tile (its
  // columns 16 .. 31, lanes g >= 2, are zeros, and so are the blocks from count on: what lies there in LDS is stale)
  auto add_zero_points = [&](int zg, int count) __attribute__((always_inline)) {
    int l = lane;
    asm volatile("" : "+v"(l));  // (what follows from the lane is computed here: the compiler would keep it in registers)
    const int r = l & 15, g = l >> 4;
    const char* const ze = smem + kZent + (zg & 1) * (kZBlocks * kEntry) + (g & 1) * (8 * kEntry) + (wave * NG * 16 + r) * 2;
    const char* const zx = smem + kZx + (((zg & 1) * BM + r) * kZBlocks + (g & 1) * 8) * 2;
    const int live = g < 2 ? count - 8 * g : 0;  // of this lane's eight blocks
    i32x4 mask;
    qmm_static_for<4>([&](auto ec) {
      constexpr int e = ec;
      mask[e] = live >= 2 * e + 2 ? -1 : live == 2 * e + 1 ? 0xffff : 0;
    });
    // (fenced off and one channel group at a time: there are few registers to spare here)
    __builtin_amdgcn_sched_barrier(0);
    qmm_static_for<NG>([&](auto gc) {
      constexpr int gi = gc;
      i32x4 za;
      qmm_static_for<4>([&](auto ec) {
        constexpr int e = ec;
        const uint32_t lo = *(const uint16_t*)(ze + (2 * e) * kEntry + gi * 32), hi = *(const uint16_t*)(ze + (2 * e + 1) * kEntry + gi * 32);
        za[e] = (int)(lo | (hi << 16)) & mask[e];
      });
      qmm_static_for<MT>([&](auto mc) {
        constexpr int mt = mc;
        const i32x4 zb = *(const i32x4*)(zx + mt * (16 * kZBlocks * 2)) & mask;
        zacc[gi][mt] = mfma16<XT>(za, zb, zacc[gi][mt]);
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };
  // Constants of the int4 expansion kept in registers the compiler cannot see through: with both constants of
  // (x & mask) | zero as literals it cannot use the single instruction for it.
  uint32_t k_zero = kInt4Bits<XT>, k_mask = kInt4Mask<XT>;
  asm volatile("" : "+v"(k_zero), "+s"(k_mask));
  // dword q (two columns) of the fragment (j, gi) of the weights in slot P (see cvt_w8 and cvt_w4)
  auto frag_q = [&](auto pc, auto jc, auto gic, auto qc) __attribute__((always_inline)) {
    constexpr int P = pc, j = jc, gi = gic, q = qc;
    if constexpr (BITS == 8) {
      return (int)cvt_w2<XT>((uint32_t)wreg[P][gi][j >> 1][(j & 1) * 2 + q / 2], qmm_const<(q & 1)>{});
    } else {
      const uint32_t d = (uint32_t)wreg[P][gi][0][j];
      constexpr int sh = XT == XLA_AMD_DT_BF16 ? 4 * q - 3 : 4 * q - 6;  // right shift (negative: left)
      const uint32_t t = sh < 0 ? d << (sh < 0 ? -sh : 0) : d >> (sh < 0 ? 0 : sh);
      return (int)((t & k_mask) | k_zero);
    }
  };
  // The weight fragments of one j (columns 32 g + 8 j .. + 7 of the step) in use and those of the next j, which are
  // converted meanwhile; the fragments of a step's first j are converted during the step before (or by prime()).
  i32x4 af[2][NG];
  auto prime = [&]() __attribute__((always_inline)) {
    qmm_static_for<NG>([&](auto gc) {
      qmm_static_for<4>([&](auto qc) { af[0][(int)gc][(int)qc] = frag_q(qmm_const<0>{}, qmm_const<0>{}, gc, qc); });
    });
  };
  // One step (128 columns), step k of LDS slot `slot`, weights in slot k % 2; `first`: it begins a block; the weights of
  // block `next` are requested into the other slot.  The order is j, row tile mt, channel group gi: an x fragment
  // serves NG MFMAs in a row and is read RX - 1 row tiles ahead into one of RX registers in turn; after every MFMA
  // its share of the next j's conversions.  A scheduling fence after each keeps that order: left to itself the
  // compiler puts the reads right before their uses and the weights' loads at the step's end.
  constexpr int RX = HASZP ? 3 : 4;
  auto compute = [&](int slot, bool first, int next, auto kc) __attribute__((always_inline)) {
    constexpr int k = kc, P = k % 2;
    load_w(next, qmm_const<1 - P>{});
    const uint32_t xt = x_at + (uint32_t)slot * (CS * X_TILE);
    const uint32_t xsq = xsq_at + (uint32_t)slot * (CS * BM * 16);
    auto xfrag = [&](int idx) __attribute__((always_inline)) {
      return *(lds_i4_t)(uintptr_t)((xt ^ (16 * (idx / MT))) + k * X_TILE + (idx % MT) * 4096);
    };
    i32x4 xq[RX];
    if constexpr (BITS == 4) {
      f32x4 q[MT];
      qmm_static_for<MT>([&](auto mc) { q[(int)mc] = *(lds_f4_t)(uintptr_t)(xsq + k * (BM * 16) + (int)mc * 256); });
      qmm_static_for<RX - 1>([&](auto ic) { xq[(int)ic] = xfrag((int)ic); });
      __builtin_amdgcn_sched_barrier(0);
      if (BLK1 || first) {
        qmm_static_for<MT>([&](auto mc) { qmm_static_for<NG>([&](auto gc) { acc[(int)gc][(int)mc] = q[(int)mc]; }); });
      } else {
        qmm_static_for<MT>([&](auto mc) { qmm_static_for<NG>([&](auto gc) { acc[(int)gc][(int)mc] += q[(int)mc]; }); });
      }
    } else {
      qmm_static_for<RX - 1>([&](auto ic) { xq[(int)ic] = xfrag((int)ic); });
      if (BLK1 || first)
        qmm_static_for<MT>([&](auto mc) { qmm_static_for<NG>([&](auto gc) { acc[(int)gc][(int)mc] = f32x4{0, 0, 0, 0}; }); });
      __builtin_amdgcn_sched_barrier(0);
    }
    qmm_static_for<4 * MT>([&](auto ic) {
      constexpr int idx = ic, j = idx / MT, mt = idx % MT;
      if constexpr (idx + RX - 1 < 4 * MT) xq[(idx + RX - 1) % RX] = xfrag(idx + RX - 1);
      qmm_static_for<NG>([&](auto gc) {
        constexpr int gi = gc, u = mt * NG + gi;
        acc[gi][mt] = mfma16<XT>(af[j & 1][gi], xq[idx % RX], acc[gi][mt]);
        constexpr int kPer = NG * 4 / (NG * MT);  // dwords of the next j's fragments per MFMA
        static_assert(kPer * MT == 4, "the conversions spread evenly over the MFMAs");
        qmm_static_for<kPer>([&](auto kc) {
          constexpr int d = u * kPer + (int)kc, gn = d / 4, q = d % 4;
          if constexpr (j < 3) af[(j + 1) & 1][gn][q] = frag_q(qmm_const<P>{}, qmm_const<(j + 1) & 3>{}, qmm_const<gn>{}, qmm_const<q>{});
          else {
            int f = frag_q(qmm_const<1 - P>{}, qmm_const<0>{}, qmm_const<gn>{}, qmm_const<q>{});
            asm volatile("" : "+v"(f));  // (here: the compiler would sink it behind the block's rounding)
            af[0][gn][q] = f;
          }
        });
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };

  // ---- results: four consecutive channels of one row per lane ----
  auto store_results = [&](const BwItem& done) __attribute__((always_inline)) {
    int l = lane;
    asm volatile("" : "+v"(l));  // (as in add_zero_points)
    const int r = l & 15, g = l >> 4;
    constexpr float kFactor = BITS == 4 ? kInt4Factor<XT> : 1.0f;
    qmm_static_for<MT>([&](auto mc) {
      constexpr int mt = mc;
      const int m = done.m0 + 16 * mt + r;
      qmm_static_for<NG>([&](auto gc) {
        constexpr int gi = gc;
        const int n = done.n0 + (wave * NG + gi) * 16 + 4 * g;
        if (m < M && n < N) {  // N % 4 == 0: the four channels exist and the address is 8-byte aligned
          float o[4];
          qmm_static_for<4>([&](auto vc) {
            constexpr int v = vc;
            float t = qmm_round_dt(kFactor * sacc[gi][mt][v], XT);
            if constexpr (HASZP) t = qmm_round_dt(t - qmm_round_dt(zacc[gi][mt][v], XT), XT);
            o[v] = t;
          });
          uint32_t lo, hi;
          if constexpr (XT == XLA_AMD_DT_BF16) {
            lo = qmm_f32x2_to_bf16x2(o[0], o[1]); hi = qmm_f32x2_to_bf16x2(o[2], o[3]);
          } else {
            lo = qmm_f32x2_to_f16x2(o[0], o[1]); hi = qmm_f32x2_to_f16x2(o[2], o[3]);
          }
          *(i32x2*)((uint16_t*)a.out + (size_t)m * N + n) = i32x2{(int)lo, (int)hi};
        }
      });
    });
  };

  int it = blockIdx.x;
  BwItem cur = item_of(it);
  set_weights(cur);
  load_w(0, qmm_const<0>{});
  int ring = 0, zg = 0;
  for (;;) {
    qmm_static_for<MT>([&](auto mc) {
      constexpr int mt = mc;
      qmm_static_for<NG>([&](auto gc) {
        sacc[(int)gc][mt] = f32x4{0, 0, 0, 0};
        zacc[(int)gc][mt] = f32x4{0, 0, 0, 0};
      });
    });
    prime();
    int s = 0, blk = 0, left = sub;  // blk: the current quantization block; left: its steps still to come
    for (int c = 0; c < n_chunks; ++c, ++ring) {
      qmm_bare_barrier();  // chunk `ring` is there (the copying waves waited for it)
      const int slot = ring & 1;
      const int s_end = min(steps, (c + 1) * CS);
      static_assert(CS % 2 == 0, "a chunk begins with weight slot 0");
      qmm_static_for<CS>([&](auto kc) {
        if (s < s_end) {
          // (the last step asks for its own weights again: never used)
          compute(slot, left == sub, min(s + 1, steps - 1), kc);
          if (BLK1 || --left == 0) {
            round_block(slot, kc);
            left = sub;
            ++blk;
            if constexpr (HASZP)
              if (blk % kZBlocks == 0) { add_zero_points(zg, kZBlocks); ++zg; }
          }
          ++s;
        }
      });
    }
    if constexpr (HASZP)
      if (blk % kZBlocks != 0) { add_zero_points(zg, blk % kZBlocks); ++zg; }

    // the next item's first weights are requested before this item's results are stored
    const BwItem done = cur;
    const int it_next = it + (int)gridDim.x;
    const bool more = it_next < n_items;
    if (more) {
      it = it_next;
      cur = item_of(it);
      set_weights(cur);
      load_w(0, qmm_const<0>{});
    }
    store_results(done);
    if (!more) break;
  }
}

template <int XT, int BITS>
int launch(const WoBwArgs& a, int cus, hipStream_t stream) {
  const int64_t items = (int64_t)((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  const dim3 grid((unsigned)(items < cus ? items : cus)), block((kComputeWaves + kCopyWaves) * 64);
  auto go = [&](auto which) -> int {
    constexpr auto kern = decltype(which)::fn;
    static std::atomic<uint64_t> lds_set{0};
    const int rc = qmm_set_max_lds((const void*)kern, kLdsBytes, lds_set, "weight_only_gemm hipFuncSetAttribute");
    if (rc != XLA_AMD_QMM_OK) return rc;
    hipLaunchKernelGGL(kern, grid, block, kLdsBytes, stream, a);
    return QMM_CHECK_LAUNCH("weight_only_gemm (blockwise, wide tile) launch");
  };
  if (!a.zp) return a.C == 128 ? go(qmm_kernel<qmm_wo_bw_wide_kernel<XT, BITS, false, true>>{}) : go(qmm_kernel<qmm_wo_bw_wide_kernel<XT, BITS, false, false>>{});
  if constexpr (BITS == 4) return go(qmm_kernel<qmm_wo_bw_wide_kernel<XT, BITS, true, true>>{});
  return qmm_fail(XLA_AMD_QMM_EUNSUPPORTED, "weight_only_gemm (blockwise, wide tile): no such kernel");
}

}  // namespace

#if QMM_WO_BW_XT == XLA_AMD_DT_BF16
int qmm_wo_bw_wide_launch_bf16(const WoBwArgs& a, int bits, int cus, hipStream_t stream) {
  return bits == 8 ? launch<XLA_AMD_DT_BF16, 8>(a, cus, stream) : launch<XLA_AMD_DT_BF16, 4>(a, cus, stream);
}
#else
int qmm_wo_bw_wide_launch_f16(const WoBwArgs& a, int bits, int cus, hipStream_t stream) {
  return bits == 8 ? launch<XLA_AMD_DT_F16, 8>(a, cus, stream) : launch<XLA_AMD_DT_F16, 4>(a, cus, stream);
}
#endif
