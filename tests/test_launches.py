"""What the library's entry points launch, recorded without a GPU."""
import ctypes
import json
import re

import pytest

from tests import launch_recorder as rec
from xla_amd import _lib, build


def test_every_kernel_gets_its_lds(tmp_path):
  """A kernel may use more than 64 KiB of dynamic LDS only once its own limit is raised: each variant of a kernel template
  behind one launcher, in one process, whatever ran before it."""
  calls = []
  for x_dt in (1, 2):
    for m, n, k, c, bits, zp in ((2048, 4096, 4096, 128, 4, True), (2048, 4096, 4096, 128, 4, False), (2048, 4096, 4096, 256, 4, False),
                                 (2048, 4096, 4096, 128, 8, False), (2048, 4096, 4096, 256, 8, False), (2048, 4096, 4096, 128, 8, True),
                                 (100, 4096, 4096, 128, 4, True), (100, 4096, 4096, 256, 4, True), (100, 4096, 4096, 128, 4, False),
                                 (100, 4096, 4096, 256, 4, False), (100, 4096, 4096, 128, 8, True), (100, 4096, 4096, 256, 8, False),
                                 (100, 4096, 4096, 4096, 8, True), (100, 4096, 4096, 4096, 8, False), (2048, 14336, 4096, 4096, 8, False),
                                 (2048, 14336, 4096, 4096, 8, True)):
      calls.append(rec.blockwise(m, n, k, c, bits, zp, x_dt))
      # scale and zero point of another dtype: the kernels whose epilogue converts at run time
      if c == k:
        name, sig, args = rec.blockwise(m, n, k, c, bits, zp, x_dt)
        calls.append((name, sig, args[:13] + [0, 0, x_dt, 0, 0] + args[-1:]))
    for zp in (True, False):
      calls += [rec.skinny(m, n, k, c, bits, zp, x_dt) for m, n, k, c, bits in
                ((4, 128256, 4096, 4096, 8), (16, 14336, 4096, 4096, 8), (32, 4096, 4096, 4096, 8), (16, 4096, 4096, 128, 4), (1, 1024, 4096, 4096, 4))]
  for out_dt in (0, 1, 2):
    calls += [rec.w8a8(m, n, 4096, out_dt=out_dt) for m, n in ((32, 4096), (512, 4096), (512, 14336), (2048, 14336), (4096, 5120))]
  seen = set()
  for call, (rc, text, launches) in zip(calls, rec.record(calls, str(tmp_path))):
    assert rc == 0 and launches, (call, text)
    for l in launches:
      seen.add(l.name)
      assert l.lds <= l.lds_limit, (l.name, l.lds, l.lds_limit)
  for kernel in ("qmm_wo_bw_wide_kernel", "qmm_wo_bw_gemm_kernel", "qmm_wo_gemm_kernel", "qmm_skinny_resident_kernel", "qmm_w8a8_gemm_kernel"):
    assert sum(kernel in s for s in seen) > 1, kernel


@pytest.mark.parametrize("zp", [False, True])
def test_row_major_rows_of_any_number(tmp_path, zp):
  """Rows past what one launch's grid can hold: pieces that follow each other and cover them all, within the limits of a
  grid (65535 in y, 2^32 threads in x)."""
  max_rows = 65535 * 64
  sizes = [(1 << 20, 8, 100), ((1 << 20) + 1, 8, 100), (max_rows, 3, 20), (max_rows + 1, 3, 20), (3 * max_rows - 5, 1, 9),
           (1, 1 << 31, 41), (5, (1 << 31) + 300, 41)]
  calls = [rec.generic(m, n, k, zp=zp) for m, n, k in sizes]
  calls += [rec.w8a8(m, n, k) for m, n, k in sizes if n <= 1 << 30]
  sizes += [s for s in sizes if s[1] <= 1 << 30]
  for (m, n, k), call, (rc, text, launches) in zip(sizes, calls, rec.record(calls, str(tmp_path))):
    assert rc == 0, (m, n, k, text)
    x_size = 2 if "generic" in call[0] else 1
    covered = {}
    for l in launches:
      assert l.grid[1] <= 65535 and l.grid[2] == 1 and l.grid[0] * l.block[0] < 1 << 32, l
      x, w, scale, _, out, lm, ln, lk = l.args
      row, col = (x - rec.PTR) // (k * x_size), (w - rec.PTR) // k
      assert lk == k and (scale - rec.PTR) == col * (2 if "generic" in call[0] else 4) and (out - rec.PTR) == (row * n + col) * 2
      # tiles of 16, 32 or 64 rows and of 16, 64 or 256 channels
      assert any(l.grid[1] == -(-lm // t) for t in (16, 32, 64)) and any(l.grid[0] == -(-ln // t) for t in (16, 64, 256))
      covered.setdefault((col, ln), []).append((row, lm))
    assert sum(ln for _, ln in covered) == n and sorted(covered)[0][0] == 0
    for rows in covered.values():
      at = 0
      for row, lm in rows:
        assert row == at
        at += lm
      assert at == m


def test_row_major_short_rows(tmp_path):
  """One thread per output up to a number of columns that depends on the outputs; its grid may be smaller than they are
  (the kernel strides) but not empty."""
  short = [(1, 1, 1), (300, 800, 16), (512, 512, 16), (513, 512, 8), (1, 32768, 40), (4, 1 << 20, 40), (1 << 20, 64, 8)]
  tiled = [(300, 800, 33), (513, 512, 9), (1, 32768, 41), (5, 65536, 9), (1, 32767, 49), (40, 3000, 2000)]
  calls = [f(*s) for f in (rec.generic, rec.w8a8) for s in short + tiled]
  calls += [rec.generic(300, 800, 17), rec.w8a8(300, 800, 31), rec.w8a8(100, 800, 47), rec.w8a8(100, 800, 49)]
  want = ([True] * len(short) + [False] * len(tiled)) * 2 + [False, True, True, False]
  for call, one_thread, (rc, text, launches) in zip(calls, want, rec.record(calls, str(tmp_path))):
    if "w8a8" in call[0] and call[2][10] % 16 == 0:
      continue  # (aligned operands take the LDS-tiled kernel)
    assert rc == 0 and len(launches) == 1, text
    assert ("qmm_rowmajor_short_kernel" in launches[0].name) == one_thread, call
    assert 0 < launches[0].grid[0] * launches[0].block[0] < 1 << 32


TILES = [(32, 32), (64, 32), (64, 64), (64, 128), (128, 128), (128, 256), (256, 256)]


def _tile(launch):
  return tuple(int(v) for v in re.search(r"qmm_w8a8_gemm_kernelILi(\d+)ELi(\d+)E", launch.name).groups())


def test_w8a8_tile_reported_is_the_tile_launched(tmp_path):
  lib, tile = _lib.load(), (ctypes.c_int32 * 3)()
  shapes = [(m, n, k) for m in (1, 32, 33, 64, 65, 128, 200, 256, 512, 1024, 2048)
            for n, k in ((1024, 4096), (4096, 4096), (4096, 14336), (14336, 4096), (28672, 4096), (8192, 1024), (5511, 4112))]
  calls = [rec.w8a8(*s) for s in shapes]
  chosen = set()
  for (m, n, k), (rc, text, launches) in zip(shapes, rec.record(calls, str(tmp_path))):
    assert rc == 0, text
    assert lib.xla_amd_qmm_w8a8_tile(m, n, k, tile) == 0
    chosen.add(tuple(tile)[:2])
    # (256 x 256 covers the last columns with tiles of 192)
    assert {_tile(l) for l in launches} <= ({(256, 256), (256, 192)} if tile[0] == 256 else {tuple(tile)[:2]}), (m, n, k)
  assert chosen == set(TILES)
  from xla_amd.experimental.hip_kernels.quantized_matmul_kernel import _SUPPORTED_TILES
  assert sorted(_SUPPORTED_TILES) == TILES
  # ... and a tile that is asked for is the one launched, at any size
  calls = [rec.w8a8(m, n, k, bm, bn) for bm, bn in TILES[:-1] for m, n, k in ((512, 4096, 4096), (10, 100, 128), (200, 4096, 14336))]
  for call, (rc, text, launches) in zip(calls, rec.record(calls, str(tmp_path))):
    assert rc == 0 and [_tile(l) for l in launches] == [tuple(call[2][-3:-1])], call


def test_quantizer_rows_of_any_number(tmp_path):
  """A grid holds fewer than 2^32 threads, whatever number of them a row gets."""
  sizes = [(m, k) for m in ((1 << 23) - 1, 1 << 23, (1 << 24) - 1) for k in (2056, 4096, 4104, 8192, 8200, 16384, 16392, 4099)]
  calls = [("xla_amd_qmm_quantize_per_token", "pppp" + "qq" + "iii" + "p", [rec.PTR, rec.PTR, rec.PTR, 0, m, k, dt, dt, 0, 0])
           for m, k in sizes for dt in (0, 1, 2)]
  for call, (rc, text, launches) in zip(calls, rec.record(calls, str(tmp_path))):
    assert rc == 0 and len(launches) == 1, (call, text)
    assert launches[0].grid[0] * launches[0].block[0] < 1 << 32, (call, launches[0])


@pytest.mark.parametrize("name,out_size", [("quantize", 1), ("dequantize", 4)])
def test_quantize_tensors_of_any_size(tmp_path, name, out_size):
  """More elements than 32-bit runs and one grid reach (an f32 result of more than 2^34 elements): pieces that follow
  each other, whichever dimension they are cut along."""
  sizes = [(1, 1, (1 << 34) + 8), (3, 1, 3 << 33), (1, 5, 7 << 32), (5, 3, (1 << 31) + 64), (1, (1 << 20) + 3, 32768)]
  calls = []
  for o, c, i in sizes:
    if name == "quantize":
      calls.append(("xla_amd_qmm_quantize_affine", "pppp" + "qqq" + "iiii" + "p", [rec.PTR, rec.PTR, rec.PTR, rec.PTR, o, c, i, 0, 0, -128, 127, 0]))
    else:
      calls.append(("xla_amd_qmm_dequantize_affine", "pppp" + "qqq" + "iii" + "p", [rec.PTR, rec.PTR, rec.PTR, rec.PTR, o, c, i, 0, 0, 1, 0]))
  in_size = 4 if name == "quantize" else 1
  for (o, c, i), (rc, text, launches) in zip(sizes, rec.record(calls, str(tmp_path))):
    assert rc == 0 and launches, text
    starts = [(l.args[0] - rec.PTR) // in_size for l in launches]
    assert starts[0] == 0 and starts == sorted(starts)
    for l, at, end in zip(launches, starts, starts[1:] + [o * c * i]):
      # a vector form, whose workgroups cover 4096 elements, or 2048 or 1024 of a short last piece
      assert "FormE3" not in l.name and l.grid[0] * l.block[0] < 1 << 32
      assert any(l.grid[0] == -(-(end - at) // n) for n in (4096, 2048, 1024)), (l, at, end)


def test_wide_tile_tests_run_the_wide_kernel(tmp_path):
  """The sizes tests/test_gpu_wo_bw_wide.py checks take the 64 x 256 tiles (the operator's counter does not tell them from
  the 64 x 128 ones), and launches of few tiles, and zero points in any other form, do not."""
  from tests.test_gpu_wo_bw_wide import test_wide_tiles
  (_, sizes), = (m.args for m in test_wide_tiles.pytestmark if m.name == "parametrize" and m.args[0].startswith("m,n,k"))
  wide = [(m, n, k, k if c == -1 else c, bits, asym) for m, n, k, c, bits, asym in sizes]
  assert len(wide) >= 9
  narrow = [(512, 4096, 4096, 128, 4, True), (100, 4096, 4096, 128, 4, False), (2048, 4096, 4096, 256, 4, True), (2048, 4096, 4096, 128, 8, True)]
  calls = [rec.blockwise(*s, x_dt) for x_dt in (1, 2) for s in wide + narrow]
  want = ["qmm_wo_bw_wide_kernel"] * len(wide) + ["qmm_wo_bw_gemm_kernel"] * len(narrow)
  for call, kernel, (rc, text, launches) in zip(calls, want * 2, rec.record(calls, str(tmp_path))):
    assert rc == 0 and len(launches) == 1 and kernel in launches[0].name, (call, text, launches)


def test_arguments_of_the_k_split_kernels():
  """The runtime writes a kernel's arguments out at every launch.  A kernel that asks for the size of its grid gets 256
  bytes of hidden ones, which made the eager call of a small launch slower than with the kernel before it."""
  with open(build.RESOURCES_PATH) as f:
    kernels = [k for k in json.load(f) if "ksplit" in k["kernel"]]
  assert len(kernels) > 50
  for k in kernels:
    assert k["kernarg_bytes"] <= 120, (k["kernel"], k["kernarg_bytes"])


def test_f32_rows_ask_for_no_workspace_they_do_not_use(tmp_path):
  """The size asked for is what the launch writes: nothing where x is multiplied as it is (and then none is needed), the
  three bf16 parts of x otherwise."""
  lib = _lib.load()
  as_it_is = [(128, 64, 128), (512, 1024, 4096), (300, 520, 640), (1, 64, 128), (128, 4096, 4096)]
  in_parts = [(2048, 4096, 4096), (256, 8192, 256), (512, 4096, 128), (1000, 14336, 4096)]
  sizes = [lib.xla_amd_qmm_weight_only_gemm_f32_workspace_bytes(*s) for s in as_it_is + in_parts]
  assert sizes == [0] * len(as_it_is) + [6 * m * k for m, _, k in in_parts]
  calls = [rec.gemm_f32(*s, workspace=0, workspace_bytes=0) for s in as_it_is]
  calls += [f(*s) for s in in_parts for f in (rec.gemm_f32, lambda *s: rec.gemm_f32(*s, workspace_bytes=6 * s[0] * s[2] - 1),
                                              lambda *s: rec.gemm_f32(*s, workspace=0))]
  got = rec.record(calls, str(tmp_path))
  for s, (rc, text, launches) in zip(as_it_is, got):
    assert rc == 0 and len(launches) == 1 and "qmm_wo_ksplit_kernel" in launches[0].name, (s, text)
  for s, (rc, text, launches), *short in zip(in_parts, *(got[len(as_it_is) + i::3] for i in range(3))):
    assert rc == 0 and ["qmm_split3_kernel" in l.name for l in launches] == [True, False], (s, text, launches)
    for rc, text, launches in short:
      assert rc != 0 and not launches and "workspace" in text, s


def _with_f32_scale(call):
  name, sig, args = call
  return (name, sig, args[:13] + [0, 0, args[15], 0, 0] + args[-1:])  # scale, zero point, result and store


def test_tiled_and_sliced_tests_run_those_kernels(tmp_path):
  """The sizes tests/test_gpu_wo_gemm.py names after a kernel run that kernel (the operator's counters count entry points,
  behind which the K split over waves takes most launches of 17 - 1000 rows)."""
  from tests.test_gpu_wo_gemm import BW_SLICED, F32_IN_PARTS, NARROW, SLICED, TILED
  calls, want = [], []
  for x_dt in (1, 2):
    for zp in (False, True):
      for m, n, k, mt, kernels in TILED:
        one = rec.blockwise(m, n, k, k, 8, zp, x_dt)
        calls += [one, _with_f32_scale(one)]
        want += [["qmm_wo_gemm_kernelILi%dELi%dE" % (x_dt, mt), "qmm_wo_gemm_finish_kernel"][:kernels]] * 2
      for m, n, k in SLICED:
        one = rec.blockwise(m, n, k, k, 8, zp, x_dt)
        calls += [one, _with_f32_scale(one)]
        want += [["qmm_skinny_kernelILi%dELi8ELi%dE" % (x_dt, 1 if m <= 16 else 2), "qmm_wo_gemm_finish_kernel"]] * 2
    for m, n, k, c, bits, zp in BW_SLICED:
      calls.append(rec.blockwise(m, n, k, c, bits, zp, x_dt))
      want.append(["qmm_skinny_kernelILi%dELi%dELi%dE" % (x_dt, bits, 1 if m <= 16 else 2), "qmm_wo_bw_finish_kernel"])
    for m, n, k, c, bits, zp in NARROW:
      calls.append(rec.blockwise(m, n, k, k if c == -1 else c, bits, zp, x_dt))
      want.append(["qmm_wo_bw_gemm_kernelILi%dELi%dELb%dELb%dE" % (x_dt, bits, zp, c == 128 and not (bits == 8 and zp))])
  for zp in (False, True):
    for s in F32_IN_PARTS:
      calls.append(rec.gemm_f32(*s, zp=zp))
      want.append(["qmm_split3_kernel", "qmm_wo_gemm_kernelILi1ELi8E"])
  seen = set()
  for call, names, (rc, text, launches) in zip(calls, want, rec.record(calls, str(tmp_path))):
    assert rc == 0 and len(launches) == len(names) and all(n in l.name for n, l in zip(names, launches)), (call[2], names, text, launches)
    seen.update(l.name for l in launches)
  # every form of the tiled kernels: 16 of the 64-row tile, 10 of the 128-row one, 14 of the blockwise one
  assert [sum(s in n for n in seen) for s in ("qmm_wo_gemm_kernelILi1ELi4E", "qmm_wo_gemm_kernelILi2ELi4E", "qmm_wo_gemm_kernelILi1ELi8E",
                                              "qmm_wo_gemm_kernelILi2ELi8E", "qmm_wo_bw_gemm_kernelI")] == [8, 8, 5, 5, 14]


def test_graph_of_workspaces_runs_two_kernels_each(tmp_path):
  from tests.test_gpu_layer import GRAPH_ROUTES
  calls = [rec.gemm_f32(m, n, k) if xdt == "f32" else rec.blockwise(m, n, k, k if c == -1 else c, 8 if c == -1 else 4, c != -1)
           for m, n, k, c, xdt in GRAPH_ROUTES]
  second = ["qmm_wo_gemm_finish_kernel", "qmm_wo_bw_finish_kernel", "qmm_wo_gemm_finish_kernel", "qmm_wo_gemm_finish_kernel",
            "qmm_wo_gemm_kernel"]
  for name, (rc, text, launches) in zip(second, rec.record(calls, str(tmp_path))):
    assert rc == 0 and len(launches) == 2 and name in launches[1].name, (text, launches)
