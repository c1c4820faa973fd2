// Matmuls against a row-major int8 weight [N, K] for any K and any alignment: the weight-only product of shapes the
// tiled copy cannot hold (K no multiple of 128) and the int8 product of activations whose K is no multiple of 16.
//
// One workgroup of eight waves owns 16 NG NW channels x 16 MT rows of x; NW waves stand side by side along the
// channels and KW = 8 / NW of them split K.  Nothing goes through LDS but the sums of the K split: a chunk of 64
// columns is 16 bytes per lane and 16 channels of weights (lane (r, g) = (lane % 16, lane / 16) takes 16 columns of row
// r) and the same columns of x, which is exactly an operand of the matrix instructions as long as both operands agree
// on the order of the columns.  Rows start at any byte: the loads are unaligned.
//
// What bounds it: memory latency at the sizes it is meant for (a few MB of weight), so a wave has the next chunk's
// loads in flight during a chunk, and few channels per workgroup put many waves on the chip.  Wide outputs with many
// rows take more channels per workgroup, since every workgroup reads its rows of x again (out of L2).
// Per launch, bf16 x against 3000 x 2000: 6.2 us for 1 row, 8.1 for 40 (one thread per output took 1060), 46 for 512.
// Then it is the loads' addresses: 40 rows took 11.0 us with 16 columns of x side by side per lane (32 bytes at a stride
// of 32, where the four lanes of a row now cover 64 consecutive bytes per load), the row's end element by element (now
// the row's last 64 columns, less those of the chunk before) and 64 rows of x loaded for 40 (now 48).  Loads two
// chunks ahead, without a branch around those past the end, made rows at odd addresses 1.5 - 3.3 times slower.
#include "qmm_common.h"
#include "qmm_frag.h"
#include "qmm_rowmajor.h"

namespace {

using namespace qmm_frag;

constexpr int kWavesAll = 8;
constexpr int kInt8 = kQmmRowMajorInt8;  // XT of the int8 product (XLA_AMD_DT_* are 0 .. 2)

template <int XT> struct Elem { typedef uint16_t t; };
template <> struct Elem<XLA_AMD_DT_F32> { typedef float t; };
template <> struct Elem<kInt8> { typedef int8_t t; };

// Result (m, n) from its sum v (f32 by bits, or int32) and, with a zero point, the row's sum of x.
template <int XT, bool HASZP>
__device__ __forceinline__ void finish_one(const QmmRowMajorArgs& a, int64_t m, int64_t n, int v, float xsum) {
  const int64_t idx = m * a.ldo + n;
  if constexpr (XT == kInt8) {
    // the chain documented at xla_amd_qmm_w8a8_gemm
    if (a.acc_out) a.acc_out[idx] = v;
    if (!a.out) return;
    float f = qmm_round_dt((float)v, a.cvt_dt);
    f = qmm_round_dt(f * qmm_load(a.scale, n, a.scale_dt), a.mid_dt);
    if (a.zp) {
      const float z = qmm_round_dt(qmm_round_dt((float)a.x_sum[m], a.zpo_dt) * qmm_load(a.zp, n, a.zp_dt), a.zpo_dt);
      f = qmm_round_dt(f - z, a.mid_dt);
    }
    qmm_store(a.out, idx, qmm_round_dt(f * qmm_load(a.x_scale, m, a.x_scale_dt), a.out_dt), a.out_dt);
  } else {
    // p = round_dot(dot); o = round_out(scale p); zero point: o = round_out(o - round_zpo(round_x(sum x) zp))
    const float p = qmm_round_dt(__int_as_float(v), a.dot_dt);
    float o = qmm_round_dt(qmm_load(a.scale, n, a.scale_dt) * p, a.out_dt);
    if constexpr (HASZP) {
      const float z = qmm_round_dt(xsum, XT) * qmm_load(a.zp, n, a.zp_dt);
      o = qmm_round_dt(o - qmm_round_dt(z, a.zpo_dt), a.out_dt);
    }
    qmm_store(a.out, idx, o, a.store_dt);
  }
}

// Rows of a few columns: one thread per output.  The tiles below load a row's end element by element under a condition
// each, and 16 rows of x whatever M is.
template <int XT, bool HASZP>
__global__ void __launch_bounds__(256)
qmm_rowmajor_short_kernel(QmmRowMajorArgs a) {
  typedef typename Elem<XT>::t elem_t;
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < a.M * a.N; idx += (int64_t)gridDim.x * 256) {
    const int64_t m = idx / a.N, n = idx - m * a.N;
    const elem_t* const x = (const elem_t*)a.x + m * a.K;
    const int8_t* const w = a.w + n * a.K;
    if constexpr (XT == kInt8) {
      int sum = 0;
      for (int k = 0; k < (int)a.K; ++k) sum += (int)x[k] * (int)w[k];
      finish_one<XT, HASZP>(a, m, n, sum, 0.f);
    } else {
      float sum = 0.f, xsum = 0.f;
      for (int k = 0; k < (int)a.K; ++k) {
        const float xv = qmm_load(x, k, XT);
        sum = fmaf(xv, (float)w[k], sum);
        if constexpr (HASZP) xsum += xv;
      }
      finish_one<XT, HASZP>(a, m, n, __float_as_int(sum), xsum);
    }
  }
}

template <int XT, int MT, int NG, int NW, bool HASZP>
__global__ void __launch_bounds__(kWavesAll * 64)
qmm_rowmajor_kernel(QmmRowMajorArgs a) {
  constexpr int KW = kWavesAll / NW;
  constexpr bool kInt = XT == kInt8;
  typedef typename Elem<XT>::t elem_t;
  constexpr int XV = (int)sizeof(elem_t);  // 16-byte pieces of a lane's 16 elements of x
  typedef i32x4 acc_t;                     // f32 or int32 sums, by bits
  __shared__ __attribute__((aligned(16))) int red[KW > 1 ? kWavesAll * (MT * NG + (HASZP ? MT : 0)) * 256 : 1];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = wave % NW, kw = wave / NW;
  const int r = lane & 15, g = lane >> 4;
  const int64_t K = a.K;
  const int64_t n0 = ((int64_t)blockIdx.x * NW + nw) * (16 * NG);
  const int64_t m0 = (int64_t)blockIdx.y * (16 * MT);

  // rows past the end read the last one again; their sums are dropped
  const int8_t* wrow[NG];
  const elem_t* xrow[MT];
  qmm_static_for<NG>([&](auto gc) { wrow[(int)gc] = a.w + min(n0 + 16 * (int)gc + r, (int64_t)a.N - 1) * K; });
  qmm_static_for<MT>([&](auto mc) { xrow[(int)mc] = (const elem_t*)a.x + min(m0 + 16 * (int)mc + r, (int64_t)a.M - 1) * K; });

  struct Chunk {
    i32x4 w[NG];
    i32x4 x[MT][XV];
  };
  // First column, within the chunk, of dword i of this lane's weights and of its x.  2-byte x takes columns 8 g .. 8 g + 7
  // of either half of the chunk, so that the four lanes of a row load 64 consecutive bytes of x; the others columns
  // 16 g .. 16 g + 15.
  constexpr bool kHalves = XV == 2;
  const int lane_col = (kHalves ? 8 : 16) * g;
  auto w_at = [](int i) constexpr { return kHalves ? 32 * (i / 2) + 4 * (i % 2) : 4 * i; };       // from there
  auto x_at = [](int i) constexpr { return kHalves ? 32 * (i / 4) + 2 * (i % 4) : 4 / XV * i; };
  constexpr bool kElements = XT == XLA_AMD_DT_F32;
  // Chunk c.  The last one ends with the row, whatever the row's length: its first columns are the chunk's before it,
  // which drop_overlap takes out.
  const int64_t last_k = K - 64;
  auto load = [&](int64_t c, Chunk& d) __attribute__((always_inline)) {
    const int64_t k = (kElements ? c * 64 : min(c * 64, last_k)) + lane_col;
    qmm_static_for<NG>([&](auto gc) {
      constexpr int gi = gc;
      if constexpr (kHalves) {
        i32x2 half[2];
        qmm_static_for<2>([&](auto hc) { __builtin_memcpy(&half[(int)hc], wrow[gi] + k + w_at(2 * (int)hc), 8); });
        d.w[gi] = i32x4{half[0][0], half[0][1], half[1][0], half[1][1]};
      } else {
        __builtin_memcpy(&d.w[gi], wrow[gi] + k, 16);
      }
    });
    qmm_static_for<MT>([&](auto mc) {
      qmm_static_for<XV>([&](auto qc) { __builtin_memcpy(&d.x[(int)mc][(int)qc], xrow[(int)mc] + k + x_at(4 * (int)qc), 16); });
    });
  };
  const int64_t chunks = (K + 63) / 64;
  const int overlap = (int)(chunks * 64 - K);
  // zeros for the columns of x in the last chunk that the one before it holds (the weights are finite)
  auto drop_overlap = [&](Chunk& d) __attribute__((always_inline)) {
    auto mask = [&](int first, int per) __attribute__((always_inline)) {  // of a dword that holds columns first .. first + per - 1
      const int k = min(max(overlap - first, 0), per);
      return k == per ? 0 : (int)(~0u << (32 / per * k));
    };
    qmm_static_for<4 * XV>([&](auto dc) {
      const int m = mask(lane_col + x_at((int)dc), 4 / XV);
      qmm_static_for<MT>([&](auto mc) { d.x[(int)mc][(int)dc / 4][(int)dc % 4] &= m; });
    });
  };
  // a chunk that the row ends in, element by element, zeros after it: the only chunk of a short row, and f32's last one
  // (there are no registers for the masks above beside f32's chunks)
  auto load_elements = [&](int64_t c, Chunk& d) __attribute__((always_inline)) {
    const int64_t k = c * 64 + lane_col;
    qmm_static_for<NG>([&](auto gc) {
      qmm_static_for<4>([&](auto dc) {
        uint32_t v = 0;
        qmm_static_for<4>([&](auto bc) {
          const int64_t at = k + w_at((int)dc) + (int)bc;
          if (at < K) v |= (uint32_t)(uint8_t)wrow[(int)gc][at] << (8 * (int)bc);
        });
        d.w[(int)gc][(int)dc] = (int)v;
      });
    });
    qmm_static_for<MT>([&](auto mc) {
      constexpr int kPer = 4 / XV;  // elements per dword
      qmm_static_for<4 * XV>([&](auto dc) {
        uint32_t v = 0;
        qmm_static_for<kPer>([&](auto bc) {
          const int64_t at = k + x_at((int)dc) + (int)bc;
          if (at < K) {
            elem_t e = xrow[(int)mc][at];
            uint32_t bits = 0;
            __builtin_memcpy(&bits, &e, sizeof(e));
            v |= bits << (8 * XV * (int)bc);
          }
        });
        d.x[(int)mc][(int)dc / 4][(int)dc % 4] = (int)v;
      });
    });
  };

  acc_t acc[NG][MT], xs[MT];
  qmm_static_for<MT>([&](auto mc) {
    xs[(int)mc] = acc_t{0, 0, 0, 0};
    qmm_static_for<NG>([&](auto gc) { acc[(int)gc][(int)mc] = acc_t{0, 0, 0, 0}; });
  });
  auto multiply = [&](const Chunk& d) __attribute__((always_inline)) {
    if constexpr (kInt) {
      qmm_static_for<NG>([&](auto gc) {
        qmm_static_for<MT>([&](auto mc) {
          acc[(int)gc][(int)mc] = __builtin_amdgcn_mfma_i32_16x16x64_i8(d.w[(int)gc], d.x[(int)mc][0], acc[(int)gc][(int)mc], 0, 0, 0);
        });
      });
    } else if constexpr (XT == XLA_AMD_DT_F32) {
      // column 16 g + t of the chunk is k = g of the t-th 16x16x4 instruction
      qmm_static_for<16>([&](auto tc) {
        constexpr int t = tc;
        qmm_static_for<MT>([&](auto mc) {
          const float xv = __int_as_float(d.x[(int)mc][t / 4][t % 4]);
          qmm_static_for<NG>([&](auto gc) {
            const float wv = (float)(int8_t)((uint32_t)d.w[(int)gc][t / 4] >> (8 * (t % 4)));
            acc[(int)gc][(int)mc] = __builtin_bit_cast(acc_t, __builtin_amdgcn_mfma_f32_16x16x4f32(
                wv, xv, __builtin_bit_cast(f32x4, acc[(int)gc][(int)mc]), 0, 0, 0));
          });
          if constexpr (HASZP)
            xs[(int)mc] = __builtin_bit_cast(acc_t, __builtin_amdgcn_mfma_f32_16x16x4f32(
                1.0f, xv, __builtin_bit_cast(f32x4, xs[(int)mc]), 0, 0, 0));
        });
      });
    } else {
      // columns 32 h + 8 g .. + 7 are the lane's eight of instruction h
      qmm_static_for<2>([&](auto hc) {
        constexpr int h = hc;
        qmm_static_for<NG>([&](auto gc) {
          const i32x4 wf = cvt_w8<XT>((uint32_t)d.w[(int)gc][2 * h], (uint32_t)d.w[(int)gc][2 * h + 1]);
          qmm_static_for<MT>([&](auto mc) {
            acc[(int)gc][(int)mc] = __builtin_bit_cast(acc_t, mfma16<XT>(wf, d.x[(int)mc][h], __builtin_bit_cast(f32x4, acc[(int)gc][(int)mc])));
          });
        });
        if constexpr (HASZP)
          qmm_static_for<MT>([&](auto mc) {
            xs[(int)mc] = __builtin_bit_cast(acc_t, mfma16<XT>(ones_frag<XT>(), d.x[(int)mc][h], __builtin_bit_cast(f32x4, xs[(int)mc])));
          });
      });
    }
  };

  auto fetch = [&](int64_t c, Chunk& d) __attribute__((always_inline)) {
    if (kElements ? c * 64 + 64 <= K : K >= 64) load(c, d);
    else load_elements(c, d);
  };
  // chunks kw, kw + KW, ...: the next one's loads are in flight during a chunk (none past the end: the loads' addresses
  // are what takes time here)
  Chunk cur;
  int64_t c = kw;
  if (c < chunks) fetch(c, cur);
  while (c < chunks) {
    Chunk next;
    const int64_t cn = c + KW;
    if (cn < chunks) fetch(cn, next);
    if constexpr (!kElements) {
      if (c == chunks - 1 && overlap > 0 && K >= 64) drop_overlap(cur);
    }
    multiply(cur);
    cur = next;
    c = cn;
  }

  // one result tile (row set gi, row tile mt): four consecutive channels of one row per lane
  auto finish = [&](int gi, int mt, acc_t v, acc_t xsum) __attribute__((always_inline)) {
    const int64_t m = m0 + 16 * mt + r, n = n0 + 16 * gi + 4 * g;
    if (m >= a.M) return;
    for (int e = 0; e < 4; ++e) {
      if (n + e >= a.N) return;
      finish_one<XT, HASZP>(a, m, n + e, v[e], __int_as_float(xsum[0]));
    }
  };
  if constexpr (KW == 1) {
    qmm_static_for<NG>([&](auto gc) {
      qmm_static_for<MT>([&](auto mc) { finish((int)gc, (int)mc, acc[(int)gc][(int)mc], xs[(int)mc]); });
    });
  } else {
    // every wave leaves its sums; wave kw then adds and finishes the tiles kw, kw + KW, ... of its channels
    constexpr int T = MT * NG, S = T + (HASZP ? MT : 0);
    i32x4* const mine = (i32x4*)red + (size_t)wave * S * 64 + lane;
    qmm_static_for<NG>([&](auto gc) {
      qmm_static_for<MT>([&](auto mc) { mine[((int)gc * MT + (int)mc) * 64] = acc[(int)gc][(int)mc]; });
    });
    if constexpr (HASZP) qmm_static_for<MT>([&](auto mc) { mine[(T + (int)mc) * 64] = xs[(int)mc]; });
    __syncthreads();
    for (int t = kw; t < T; t += KW) {
      acc_t v = {0, 0, 0, 0}, xv = {0, 0, 0, 0};
      auto add = [&](acc_t& to, int slot) __attribute__((always_inline)) {
        for (int k2 = 0; k2 < KW; ++k2) {
          const acc_t o = ((const i32x4*)red)[((size_t)(k2 * NW + nw) * S + slot) * 64 + lane];
          if constexpr (kInt) to += o;
          else to = __builtin_bit_cast(acc_t, __builtin_bit_cast(f32x4, to) + __builtin_bit_cast(f32x4, o));
        }
      };
      add(v, t);
      if constexpr (HASZP) add(xv, T + t % MT);
      finish(t / MT, t % MT, v, xv);
    }
  }
}

template <int XT, int MT, int NG, int NW>
int launch(const QmmRowMajorArgs& a, hipStream_t stream) {
  constexpr int BN = 16 * NG * NW, BM = 16 * MT;
  const dim3 grid((unsigned)((a.N + BN - 1) / BN), (unsigned)((a.M + BM - 1) / BM)), block(kWavesAll * 64);
  if (XT != kInt8 && a.zp) hipLaunchKernelGGL((qmm_rowmajor_kernel<XT, MT, NG, NW, XT != kInt8>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((qmm_rowmajor_kernel<XT, MT, NG, NW, false>), grid, block, 0, stream, a);
  return QMM_CHECK_LAUNCH("row-major matmul launch");
}

// Channels per workgroup: 256 (every wave its own 32) where that still is two workgroups per compute unit (f32 x, 2048
// rows against 3000 x 2000, which is 384 of them: 342 us so, 291 with 64 channels), 64 (two waves side by side, four
// along K) where that fills most of the chip once (512 rows of bf16: 46 us, 52 with 16 channels), else 16 (all eight
// waves along K: it takes that many waves to have a few MB of weight in flight).
template <int XT, int MT>
int launch_width(const QmmRowMajorArgs& a, hipStream_t stream) {
  const int64_t row_tiles = (a.M + 16 * MT - 1) / (16 * MT);
  if ((int64_t)((a.N + 255) / 256) * row_tiles >= 512) return launch<XT, MT, 2, 8>(a, stream);
  if ((int64_t)((a.N + 63) / 64) * row_tiles >= 200) return launch<XT, MT, 2, 2>(a, stream);
  return launch<XT, MT, 1, 1>(a, stream);
}

// Columns up to which one thread per output is faster (bf16 x / int8 x, us, one thread per output against tiles): the
// latency of its loop decides for few outputs (512 x 512: K = 12 6.0 / 4.7 against 7.3 / 8.6, K = 25 9.1 / 8.3 against
// 7.9 / 9.5, K = 33 12.1 / 11.1 against 8.0 / 9.7; 40 x 3000: K = 12 5.3 / 3.9 against 7.0 / 8.4, K = 40 11.7 / 7.5
// against 7.7 / 9.4, K = 50 14.3 / 9.0 against 7.8 / 9.5), its many loads for many (2048 x 2048: K = 4 24 / 17 against
// 32 / 24, K = 8 33 / 23 against 35 / 25, K = 12 42 / 32 against 38 / 27), and the tiles' empty rows for one row against
// many channels (1 x 1 048 576: K = 8 11 / 8 against 40 / 56, K = 40 62 / 61 against 65 / 79).
inline int64_t short_columns(const QmmRowMajorArgs& a, bool int8) {
  if (a.M <= 4 && a.N >= 32768) return 40;
  if (a.M * a.N > (1 << 18)) return 8;
  return !int8 ? 16 : a.M * a.N > (1 << 17) ? 32 : 48;
}

template <int XT>
int launch_rows(const QmmRowMajorArgs& a, hipStream_t stream) {
  if (a.K <= short_columns(a, XT == kInt8)) {
    const int64_t blocks = (a.M * a.N + 255) / 256;
    const dim3 grid((unsigned)(blocks < 65536 ? blocks : 65536)), block(256);
    if (XT != kInt8 && a.zp) hipLaunchKernelGGL((qmm_rowmajor_short_kernel<XT, XT != kInt8>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((qmm_rowmajor_short_kernel<XT, false>), grid, block, 0, stream, a);
    return QMM_CHECK_LAUNCH("row-major matmul launch");
  }
  if (a.M <= 16) return launch_width<XT, 1>(a, stream);
  if (a.M <= 32) return launch_width<XT, 2>(a, stream);
  if (a.M <= 48) return launch_width<XT, 3>(a, stream);
  return launch_width<XT, 4>(a, stream);
}

}  // namespace

static int launch_piece(const QmmRowMajorArgs& a, int x_dt, hipStream_t stream) {
  switch (x_dt) {
    case XLA_AMD_DT_F32: return launch_rows<XLA_AMD_DT_F32>(a, stream);
    case XLA_AMD_DT_BF16: return launch_rows<XLA_AMD_DT_BF16>(a, stream);
    case XLA_AMD_DT_F16: return launch_rows<XLA_AMD_DT_F16>(a, stream);
    default: return launch_rows<kInt8>(a, stream);
  }
}

// What one grid cannot hold goes in pieces: 65535 tiles of 64 rows, and channels whose tiles come to less than 2^32
// threads.
int qmm_rowmajor_launch(const QmmRowMajorArgs& whole, int x_dt, hipStream_t stream) {
  constexpr int64_t kRows = 65535ll * 64, kChannels = 1ll << 30;
  if ((whole.M * whole.N + 255) / 256 > 0x7fffffffLL) return qmm_fail(XLA_AMD_QMM_EUNSUPPORTED, "row-major matmul: too many outputs");
  const bool int8 = x_dt == kInt8;
  const size_t x_size = int8 ? 1 : qmm_dt_size(x_dt), out_size = qmm_dt_size(int8 ? whole.out_dt : whole.store_dt);
  auto at = [](const void* p, int64_t elements, size_t size) { return p ? (void*)((char*)p + elements * size) : nullptr; };
  for (int64_t n = 0; n < whole.N; n += kChannels) {
    for (int64_t m = 0; m < whole.M; m += kRows) {
      QmmRowMajorArgs a = whole;
      a.ldo = whole.N;
      a.M = whole.M - m < kRows ? whole.M - m : kRows;
      a.N = whole.N - n < kChannels ? whole.N - n : kChannels;
      a.x = at(whole.x, m * whole.K, x_size);
      a.w = whole.w + n * whole.K;
      a.scale = at(whole.scale, n, qmm_dt_size(whole.scale_dt));
      a.zp = at(whole.zp, n, qmm_dt_size(whole.zp_dt));
      a.out = at(whole.out, m * whole.N + n, out_size);
      a.x_scale = at(whole.x_scale, m, qmm_dt_size(whole.x_scale_dt));
      a.x_sum = (const int32_t*)at(whole.x_sum, m, 4);
      a.acc_out = (int32_t*)at(whole.acc_out, m * whole.N + n, 4);
      const int rc = launch_piece(a, x_dt, stream);
      if (rc != XLA_AMD_QMM_OK) return rc;
    }
  }
  return XLA_AMD_QMM_OK;
}
