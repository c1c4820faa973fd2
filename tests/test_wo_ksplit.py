"""Batches of rows against per-channel int8 weights: K split over the waves of a workgroup, one shape or more per tile."""
import re

import pytest
import torch

from oracle import quantized_matmul_oracle as oracle
from tests import cases
from tests import launch_recorder as rec

# (m, n, k, rows and channels of the tile): row tiles of unequal length, a last tile of few rows and of few channels, n
# that is and is not a multiple of 4 (channel groups of 10, 12, 14 and 16), k of less than a slot, of one, and of several
# with a last one that not every wave has a share of
SHAPES = [
    (17, 16, 128, 16, 16), (31, 30, 2176, 16, 16), (129, 17, 1152, 16, 16),
    (17, 2049, 640, 16, 32), (128, 520, 2176, 16, 32),
    (17, 2049, 128, 32, 32), (32, 6146, 384, 32, 32), (193, 1030, 512, 32, 32),
    (97, 2049, 128, 32, 64), (64, 7165, 384, 32, 64), (511, 1000, 640, 32, 64),
    (33, 4100, 128, 48, 32), (97, 2049, 1152, 48, 32),
    (129, 4100, 128, 48, 64), (100, 4100, 2176, 48, 64),
    (65, 6146, 128, 64, 64), (385, 2049, 640, 64, 64),
    (129, 7165, 128, 64, 96), (250, 5000, 640, 64, 96),
    (193, 6146, 128, 64, 128), (300, 6146, 1152, 64, 128), (2048, 1000, 640, 64, 128),
]


# f32 rows: from one; a tile of 16 x 16 with four and with eight K groups
F32_SHAPES = [
    (1, 5, 128, 16, 16), (17, 333, 384, 16, 16), (1, 5, 640, 16, 16), (127, 333, 2176, 16, 16),
    (1, 4100, 640, 16, 32), (100, 4100, 640, 16, 32),
    (33, 4100, 2176, 16, 64), (100, 2049, 640, 16, 64),
    (17, 4100, 384, 32, 32), (127, 1030, 128, 32, 32),
    (33, 7165, 128, 32, 64), (127, 7165, 1152, 32, 64),
    (300, 520, 640, 32, 32),  # more rows than the streaming kernel gets
]


# blockwise and int4 weights (m, n, k, c, bits, zero point, rows and channels of the tile): c = -1 is per-channel; blocks of
# one, two, three and five tiles of 128 columns; fewer blocks than K groups, and a last round that not every group has
BW_SHAPES = [
    (17, 20, 256, 128, 4, True, 16, 16), (64, 132, 2176, 128, 8, True, 16, 16), (33, 100, 1920, 640, 4, False, 16, 16),
    (17, 2300, 2304, 256, 4, False, 16, 32), (100, 1024, 1152, 128, 4, True, 16, 32),
    (32, 5000, 384, 384, 4, True, 32, 32), (64, 4096, 1152, 128, 8, False, 32, 32), (40, 4100, 2560, 256, 8, True, 48, 32),
    (65, 4096, 1280, 128, 4, True, 48, 32), (48, 6144, 640, -1, 4, True, 48, 32),
    (48, 12000, 1152, 128, 4, True, 48, 64), (96, 6000, 768, 256, 8, False, 48, 64),
    (128, 4096, 640, 128, 4, True, 64, 32), (200, 2048, 1152, -1, 4, False, 64, 32),
    (200, 4096, 1152, 128, 4, False, 64, 64), (250, 4000, 1536, 512, 8, False, 64, 64),
]


def test_tiles_of_the_blockwise_shapes(tmp_path):
  calls = [rec.blockwise(m, n, k, k if c == -1 else c, bits, zp, dt) for m, n, k, c, bits, zp, _, _ in BW_SHAPES for dt in (1, 2)]
  calls += [rec.skinny(m, n, k, k if c == -1 else c, bits, zp, 1) for m, n, k, c, bits, zp, _, _ in BW_SHAPES if m <= 64]
  want = {(m, n, k): (bm, bn) for m, n, k, _, _, _, bm, bn in BW_SHAPES}
  got = {}
  for (_, _, args), (rc, text, launches) in zip(calls, rec.record(calls, str(tmp_path))):
    assert rc == 0, text
    m, n, k = args[7:10] if len(args) > 18 else args[5:8]
    (l,) = launches
    mt, ng, kw, cw = (int(v) for v in re.search(r"_ksplitILi\dELi\dELi(\d)ELi(\d)ELi(\d)ELi(\d)E", l.name).groups())
    assert l.lds <= l.lds_limit and l.block[0] == 64 * (kw * cw + 4)
    got[m, n, k] = (16 * mt, 16 * ng * cw)
  assert got == want
  assert len(set(want.values())) == 7
  # scales of another dtype, 16 rows or fewer and wide outputs of up to 64 keep the streaming kernel
  name, sig, args = rec.skinny(40, 64, 256, 256, 4, False, 1)
  calls = [(name, sig, args[:11] + [0, 1, 1, 0, 0] + args[-1:]), rec.skinny(16, 2048, 2048, 128, 4, True), rec.skinny(64, 32768, 1024, 128, 4, True)]
  for rc, text, launches in rec.record(calls, str(tmp_path)):
    assert rc == 0 and launches and not any("ksplit" in l.name for l in launches), text


def test_blockwise_launches_left_to_the_older_kernels(tmp_path):
  """Blockwise launches that are shorter in K slices of the streaming kernel, in one pass of it, or in the tiles of the GEMM,
  beside ones of the same kinds that are not."""
  want = [
      # K slices: 17 - 32 rows, few channels, a long K in long blocks
      ((27, 620, 13312, 512, 8, False), "qmm_skinny_kernel"), ((17, 256, 16384, 256, 8, False), "qmm_skinny_kernel"),
      ((24, 1536, 10240, 1024, 8, False), "qmm_skinny_kernel"), ((18, 4168, 11264, 512, 4, False), "qmm_skinny_kernel"),
      ((32, 512, 4096, 128, 4, False), "ksplit"), ((24, 512, 14336, -1, 4, True), "ksplit"), ((32, 4096, 4096, 128, 4, True), "ksplit"),
      # two long blocks
      ((18, 4892, 1024, 512, 4, True), "qmm_skinny_kernel"), ((20, 1024, 2048, 1024, 8, False), "qmm_skinny_kernel"),
      ((18, 4892, 1024, 128, 4, True), "ksplit"), ((20, 1024, 4096, 1024, 8, False), "ksplit"),
      # tiles of the GEMM
      ((314, 8176, 12800, 128, 4, False), "qmm_wo_bw_wide_kernel"), ((603, 4308, 13824, 128, 4, False), "qmm_wo_bw_wide_kernel"),
      ((629, 3224, 7936, 128, 4, True), "qmm_wo_bw_wide_kernel"), ((633, 4224, 10240, 512, 8, False), "qmm_wo_bw_wide_kernel"),
      ((128, 4096, 4096, 128, 4, True), "ksplit"), ((300, 2048, 8192, 256, 4, False), "ksplit"), ((100, 4096, 8192, 128, 8, False), "ksplit"),
  ]
  calls = [(rec.skinny if m <= 32 and k < 4096 else rec.blockwise)(m, n, k, k if c == -1 else c, bits, zp, dt)
           for (m, n, k, c, bits, zp), _ in want for dt in (1, 2)]
  for (shape, kernel), got in zip([w for w in want for _ in (1, 2)], rec.record(calls, str(tmp_path))):
    rc, text, launches = got
    assert rc == 0 and kernel in launches[0].name, (shape, text, launches)
  # without the workspace that the slices need, the split takes them
  name, sig, args = rec.blockwise(27, 620, 13312, 512, 8, False)
  ((rc, text, launches),) = rec.record([(name, sig, args[:5] + [0, 0] + args[7:])], str(tmp_path))
  assert rc == 0 and "ksplit" in launches[0].name, text


def test_many_rows_against_few_channels(tmp_path):
  """More rows than the estimates were fitted to: the reads of x decide."""
  want = [((5650, 317, 7936, -1, 8, False), "qmm_wo_gemm_kernel"), ((2557, 949, 13952, -1, 8, False), "qmm_wo_gemm_kernel"),
          ((2048, 1000, 640, -1, 8, True), "ksplit"), ((1500, 600, 4096, -1, 8, False), "ksplit"),
          ((3956, 196, 3200, -1, 4, True), "qmm_wo_bw_gemm_kernelI"), ((6234, 156, 3584, 512, 4, True), "qmm_wo_bw_gemm_kernelI"),
          ((1927, 492, 1408, 128, 8, True), "qmm_wo_bw_gemm_kernelI"), ((1200, 512, 4096, 128, 4, True), "ksplit")]
  calls = [rec.blockwise(m, n, k, k if c == -1 else c, bits, zp, dt) for (m, n, k, c, bits, zp), _ in want for dt in (1, 2)]
  for (shape, kernel), (rc, text, launches) in zip([w for w in want for _ in (1, 2)], rec.record(calls, str(tmp_path))):
    assert rc == 0 and kernel in launches[0].name, (shape, text, launches)


def test_tiles_of_the_f32_shapes(tmp_path):
  calls = [rec.skinny(m, n, k, k, 8, zp, 0) for m, n, k, _, _ in F32_SHAPES for zp in (False, True)]
  seen = set()
  for (_, _, args), (rc, text, launches) in zip(calls, rec.record(calls, str(tmp_path))):
    assert rc == 0, text
    m, n, k = args[5:8]
    (l,) = launches
    xt, mt, ng, kw, cw = (int(v) for v in re.search(r"qmm_wo_ksplit_kernelILi(\d)ELi(\d)ELi(\d)ELi(\d)ELi(\d)E", l.name).groups())
    assert xt == 0 and (m, n, k, 16 * mt, 16 * ng * cw) in F32_SHAPES, (m, n, k, l.name)
    assert l.lds <= l.lds_limit and l.block[0] == 64 * (kw * cw + 4)
    seen.add((mt, ng, kw, cw))
  assert len(seen) == 6
  # rows that fill the chip keep the split into three bf16 parts, sizes past the kernel's range the streaming kernel
  calls = [rec.skinny(4, 64, 131072, 131072, 8, False, 0), rec.skinny(16, 16384, 640, 640, 8, False, 0),
           ("xla_amd_qmm_weight_only_gemm_f32", "pppppp" + "z" + "qqq" + "iip", [rec.PTR] * 3 + [0, rec.PTR, rec.PTR, 1 << 40, 2048, 4096, 4096, 0, 0, 0])]
  for rc, text, launches in rec.record(calls, str(tmp_path)):
    assert rc == 0 and launches and not any("ksplit" in l.name for l in launches), text


def test_f32_rows_against_wide_outputs(tmp_path):
  """17 - 127 rows against many channels and a short K: a pass of the streaming kernel per 16 rows where a third, fifth or
  seventh one is shorter than a row tile of 32 for the last of them, K split over waves otherwise."""
  stream = [(33, 128256, 384), (48, 65536, 128), (33, 32768, 640), (65, 128256, 768), (97, 128256, 640), (17, 262144, 640)]
  split = [(33, 16384, 384), (49, 128256, 384), (33, 32768, 512), (64, 128256, 768), (127, 128256, 640), (32, 128256, 512),
           (33, 128256, 1152), (100, 128256, 4096), (127, 1 << 19, 2048)]
  calls = [rec.skinny(m, n, k, k, 8, zp, 0) for m, n, k in stream + split for zp in (False, True)]
  for (_, _, args), (rc, text, launches) in zip(calls, rec.record(calls, str(tmp_path))):
    assert rc == 0, text
    m, n, k = args[5:8]
    if (m, n, k) in stream:
      assert len(launches) == -(-m // 16) and all("qmm_skinny_kernel" in l.name for l in launches), (m, n, k, launches)
    else:
      assert len(launches) == 1 and "qmm_wo_ksplit_kernel" in launches[0].name, (m, n, k, launches)


def test_tiles_of_the_shapes(tmp_path):
  calls = [rec.blockwise(m, n, k, k, 8, zp, dt) for m, n, k, _, _ in SHAPES for zp in (False, True) for dt in (1, 2)]
  calls += [rec.skinny(m, n, k, k, 8, zp, 1) for m, n, k, _, _ in SHAPES if m <= 32 for zp in (False, True)]
  want = {(m, n, k): (bm, bn) for m, n, k, bm, bn in SHAPES}
  seen = set()
  for (_, sig, args), (rc, text, launches) in zip(calls, rec.record(calls, str(tmp_path))):
    assert rc == 0, text
    m, n, k = args[7:10] if len(args) > 18 else args[5:8]
    (l,) = launches
    mt, ng, kw, cw = (int(v) for v in re.search(r"qmm_wo_ksplit_kernelILi\dELi(\d)ELi(\d)ELi(\d)ELi(\d)E", l.name).groups())
    assert (16 * mt, 16 * ng * cw) == want[m, n, k], (m, n, k, l.name)
    tiles = -(-m // (16 * mt)) * -(-n // (16 * ng * cw))
    assert l.lds <= l.lds_limit and l.block[0] == 64 * (kw * cw + 4) and tiles <= l.grid[0] < tiles + 8, l
    seen.add(want[m, n, k])
  assert len(seen) == 9
  # 16 rows or fewer, and wide outputs of up to 32, keep the streaming kernel; what fills the chip keeps the tiled GEMM
  calls = [rec.skinny(16, 4096, 4096, 4096, 8, False), rec.skinny(32, 14336, 4096, 4096, 8, False),
           rec.blockwise(2048, 14336, 4096, 4096, 8, False)]
  for rc, text, launches in rec.record(calls, str(tmp_path)):
    assert rc == 0 and not any("ksplit" in l.name for l in launches), text


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,bm,bn", SHAPES)
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16])
def test_against_the_oracle(m, n, k, bm, bn, xdt):
  import xla_amd.experimental.custom_kernel  # noqa: F401
  op = torch.ops.xla.quantized_matmul
  for zp, sdt in ((False, torch.float32), (False, xdt), (True, xdt), (True, torch.float32)):
    x, w, s, _ = cases.per_channel_int8(m, n, k, xdt, sdt, seed=m + n)
    z = (torch.randn(n, generator=cases.gen(5)) * 0.01).to(sdt) if zp else None
    exp = oracle.quantized_matmul(x, w, s, z)
    wd, sd, zd = w.cuda(), s.cuda(), None if z is None else z.cuda()
    out = op(x.cuda(), wd, sd, zd).cpu()
    # f32 sums in another order: a dot product rounds to its other neighbour now and then
    assert out.dtype == exp.dtype and cases.within_tolerance(out, exp), (zp, sdt)
    assert cases.rel_l2(out, exp) < 1e-3, (zp, sdt)
  # an infinity stays in its row: the other rows of the tile, and of the row quad copied with it, are untouched
  row = m - 1
  x[row, 3] = float("inf")
  bad = op(x.cuda(), wd, sd, zd).cpu()
  assert torch.equal(bad[:row], out[:row])
  assert not torch.isfinite(bad[row]).any()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,bm,bn", F32_SHAPES + [(33, 32768, 640, 16, 64)])  # (the last: three passes of the streaming kernel)
def test_f32_against_f64(m, n, k, bm, bn):
  import xla_amd.experimental.custom_kernel  # noqa: F401
  op = torch.ops.xla.quantized_matmul
  for zp, sdt in ((False, torch.bfloat16), (False, torch.float32), (True, torch.float32), (True, torch.bfloat16)):
    x, w, s, _ = cases.per_channel_int8(m, n, k, torch.float32, sdt, seed=m + n)
    z = (torch.randn(n, generator=cases.gen(5)) * 0.01).to(sdt) if zp else None
    exp = (x.double() @ w.double().T) * s.double()
    mag = (x.double().abs() @ w.double().abs().T) * s.double().abs()
    if zp:
      exp -= x.double().sum(1, keepdim=True) * z.double()
      mag += x.double().abs().sum(1, keepdim=True) * z.double().abs()
    wd, sd, zd = w.cuda(), s.cuda(), None if z is None else z.cuda()
    out = op(x.cuda(), wd, sd, zd).cpu()
    # products, sums and the few operations behind them, each within half an ulp of what it handles
    assert out.dtype == torch.float32 and ((out.double() - exp).abs() <= (k / 2 + 8) * 2.0**-24 * mag).all(), (zp, sdt)
    assert cases.rel_l2(out, exp) < 1e-5, (zp, sdt)
  row = m - 1
  x[row, 3] = float("inf")
  bad = op(x.cuda(), wd, sd, zd).cpu()
  assert torch.equal(bad[:row], out[:row])
  assert not torch.isfinite(bad[row]).any()


# past the K of this kernel the streaming kernel runs, with one and two x tiles and K split over four waves
LONG_ROWS = [(8, 61, 66048, torch.float32), (20, 61, 66048, torch.bfloat16), (20, 61, 66048, torch.float16)]


def test_long_rows_keep_the_streaming_kernel(tmp_path):
  dts = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}
  calls = [rec.skinny(m, n, k, k, 8, zp, dts[xdt]) for m, n, k, xdt in LONG_ROWS for zp in (False, True)]
  for call, (rc, text, launches) in zip(calls, rec.record(calls, str(tmp_path))):
    assert rc == 0 and len(launches) == 1, text
    assert re.search(r"qmm_skinny_kernelILi\dELi8ELi%dELi4ELi1E" % (2 if call[2][5] > 16 else 1), launches[0].name), launches


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,xdt", LONG_ROWS)
def test_long_rows(m, n, k, xdt):
  import xla_amd.experimental.custom_kernel  # noqa: F401
  for zp, sdt in ((False, xdt), (True, xdt), (False, torch.float32), (True, torch.float32)):
    x, w, s, _ = cases.per_channel_int8(m, n, k, xdt, sdt, seed=m)
    z = (torch.randn(n, generator=cases.gen(5)) * 0.01).to(sdt) if zp else None
    exp = oracle.quantized_matmul(x, w, s, z)
    out = torch.ops.xla.quantized_matmul(x.cuda(), w.cuda(), s.cuda(), None if z is None else z.cuda()).cpu()
    assert out.dtype == exp.dtype and cases.within_tolerance(out, exp) and cases.rel_l2(out, exp) < 1e-3, (zp, sdt)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,c,bits,zp,bm,bn", BW_SHAPES)
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16])
def test_blockwise_against_the_oracle(m, n, k, c, bits, zp, bm, bn, xdt):
  import xla_amd.experimental.custom_kernel  # noqa: F401
  op = torch.ops.xla.quantized_matmul
  if c == -1:
    x, w, s, _ = cases.per_channel_int8(m, n, k, xdt, xdt, seed=m)
    w, z = w.clamp(-8, 7), (torch.randn(n, generator=cases.gen(5)) * 0.01).to(xdt)
  else:
    x, w, s, z, _ = cases.blockwise(m, n, k, c, bits, xdt, symmetric=not zp, seed=m + k)
  z = z if zp else None
  exp = oracle.quantized_matmul(x, w, s, z, block_size=c, int4_weight=bits == 4)
  wd, sd, zd = w.cuda(), s.cuda(), None if z is None else z.cuda()
  out = op(x.cuda(), wd, sd, zd, c, bits == 4).cpu()
  # f32 sums in another order: a dot product rounds to its other neighbour now and then (the bound of the tiled GEMM)
  assert out.dtype == exp.dtype and cases.within_tolerance(out, exp)
  assert cases.rel_l2(out, exp) < 1e-3
  x[m - 1, 3] = float("inf")
  bad = op(x.cuda(), wd, sd, zd, c, bits == 4).cpu()
  assert torch.equal(bad[:m - 1], out[:m - 1])
  assert not torch.isfinite(bad[m - 1]).any()


@pytest.mark.gpu
def test_replays_and_streams():
  """No workspace, no state: replays of a captured launch and launches on two streams at once give the same results."""
  import xla_amd.experimental.custom_kernel  # noqa: F401
  op = torch.ops.xla.quantized_matmul
  x, w, s, _ = cases.per_channel_int8(100, 2049, 1152, torch.bfloat16, torch.bfloat16, seed=1)
  x, w, s = x.cuda(), w.cuda(), s.cuda()
  ref = op(x, w, s)
  torch.cuda.synchronize()
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    out = op(x, w, s)
  for _ in range(4):
    out.zero_()
    graph.replay()
    assert torch.equal(op(x, w, s), ref)
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
  streams = [torch.cuda.Stream() for _ in range(2)]
  outs = []
  for _ in range(8):
    for st in streams:
      with torch.cuda.stream(st):
        outs.append(op(x, w, s))
  torch.cuda.synchronize()
  assert all(torch.equal(o, ref) for o in outs)
