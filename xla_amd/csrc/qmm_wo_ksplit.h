// The parts that the kernels with K split over the waves of a workgroup share (qmm_wo_ksplit.hip, per-channel weights;
// qmm_wo_ksplit_bw.hip, blockwise and int4 weights): shape of a workgroup, its tile, and the copying waves.
#pragma once
#include "qmm_common.h"
#include "qmm_frag.h"
#include "qmm_wo_gemm.h"

namespace {

using namespace qmm_frag;

constexpr int kCopyWaves = 4;
constexpr int kLds = 160 * 1024;

// The launch's tiles.  (All that a kernel needs to know of its grid, see KsArgs.)
inline KsTiles ks_tiles(int M, int N, int bm, int bn) {
  KsTiles t;
  t.tiles_m = (M + bm - 1) / bm;
  t.rows = (M + t.tiles_m - 1) / t.tiles_m;
  t.tiles = t.tiles_m * ((N + bn - 1) / bn);
  t.per_xcd = (t.tiles + 7) / 8;
  t.tiles_m_magic = (((uint64_t)1 << 32) + t.tiles_m - 1) / t.tiles_m;
  return t;
}

// TAIL: bytes of LDS beside the ring and, after it, the partial sums.
template <int XT, int MT, int NG, int KW, int CW, int TAIL> struct KsCfg {
  static constexpr int NW = KW * CW;             // computing waves
  static constexpr int BM = 16 * MT, BN = 16 * NG * CW;
  static constexpr int ROW = XT == XLA_AMD_DT_F32 ? 512 : 256;  // bytes of one row of a tile (128 columns of x)
  static constexpr int TILE = BM * ROW;
  static constexpr int SLOT = KW * TILE;
  static constexpr int PITCH = BN + 4;           // floats per row of the partial sums (4 more: rows start on other banks)
  static constexpr int kSums = KW * BM * (PITCH + 1) * 4;  // partial sums, and partial row sums of x
  static constexpr int kFit = (kLds - TAIL) / SLOT;
  static constexpr int R = kFit < 8 ? kFit : 8;  // slots of the ring
  static_assert(R >= 2, "the ring needs room to run ahead");
  static constexpr int lds_bytes(int steps) {
    const int ring = (steps < R ? steps : R) * SLOT;
    return TAIL + (ring > kSums ? ring : kSums);
  }
  static_assert(TAIL + kSums <= kLds, "the partial sums fit");
};

// The tile of this workgroup: first channel and row, live rows; false if there is none.  Workgroups are dealt round-robin
// to the 8 XCDs: each XCD gets a contiguous run of the tiles, row tiles fastest, so that the row tiles of a column share
// its weights in that L2 (tile / tiles_m by multiply-shift: tile < 2^16).
__device__ __forceinline__ bool ks_tile_of(const KsTiles& t, int M, int bn, int& n0, int& m0, int& rows) {
  const int tile = ((int)blockIdx.x & 7) * t.per_xcd + ((int)blockIdx.x >> 3);
  if (tile >= t.tiles) return false;
  const int col = (int)(((uint64_t)(uint32_t)tile * t.tiles_m_magic) >> 32);
  n0 = col * bn;
  m0 = (tile - col * t.tiles_m) * t.rows;
  rows = min(t.rows, M - m0);
  return true;
}

// Copying wave cw: the x tiles of all slots, KW per slot (tile_of(slot, k): the k th), R - 1 slots ahead of the
// computing waves, which it meets once per slot and once more when they have read the last one.  ahead() runs between
// the first slots' copies and the rest, behind() before that last meeting.
template <class Cfg, int KW, class TileOf, class Ahead, class Behind>
__device__ __forceinline__ void ks_copy_x(const void* x, int K, int m0, int rows, int steps, int cw, int lane, char* ring,
                                          TileOf&& tile_of, Ahead&& ahead_of_loop, Behind&& behind_loop) {
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  constexpr int R = Cfg::R, D = R - 1, TILE = Cfg::TILE, SLOT = Cfg::SLOT;
  constexpr int kRows = 1024 / Cfg::ROW;               // rows per instruction
  constexpr int kLanes = 64 / kRows;                   // lanes per row
  constexpr int L = Cfg::BM / kRows / kCopyWaves;      // instructions per wave and tile
  const int pieces = (rows + kRows - 1) / kRows;
  const int nq = pieces > cw ? (pieces - cw + kCopyWaves - 1) / kCopyWaves : 0;  // of this wave: cw, cw + 4, ...
  const char* const xb = (const char*)x + (size_t)m0 * K * (Cfg::ROW / 128);
  uint32_t x_off[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int row = min((cw + i * kCopyWaves) * kRows + lane / kLanes, rows - 1);
    x_off[i] = (uint32_t)row * ((uint32_t)K * (Cfg::ROW / 128)) + (uint32_t)(((lane % kLanes) ^ (row & 15)) * 16);
  }
  int issued = 0, slot = 0;
  auto issue = [&]() __attribute__((always_inline)) {
    char* const dst = ring + slot * SLOT;
#pragma unroll
    for (int k = 0; k < KW; ++k) {
      const char* const src = xb + (size_t)tile_of(issued, k) * Cfg::ROW;
#pragma unroll
      for (int i = 0; i < L; ++i)
        if (i < nq)
          __builtin_amdgcn_global_load_lds((const void*)(src + (size_t)x_off[i]), (lds_ptr_t)(dst + k * TILE + (cw + i * kCopyWaves) * 1024), 16, 0, 0);
    }
    ++issued;
    slot = slot + 1 == R ? 0 : slot + 1;
  };
  while (issued < min(D, steps)) issue();
  ahead_of_loop();
  for (int n = 0; n < steps; ++n) {
    // the loads of the slots after n may be in flight (a wave's loads complete in order)
    const int ahead = issued - 1 - n;
    bool done = false;
    qmm_static_for<D>([&](auto dc) {
      qmm_static_for<L + 1>([&](auto qc) {
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
  behind_loop();
  qmm_bare_barrier();  // the computing waves have read the last slot
}

}  // namespace
