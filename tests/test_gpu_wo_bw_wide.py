"""Blockwise and int4 weights against many rows: launches large enough for the 64 x 256 tiles, against the oracle."""
import pytest
import torch

from oracle import quantized_matmul_oracle as oracle
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
  import xla_amd.experimental.xla_quantized_matmul as q
  return q


# 1030 rows x 2052 channels are 289 tiles of 64 x 128 (two rounds over 256 compute units) and 153 of 64 x 256 (one),
# the last of 6 rows and of 4 channels; 2050 x 4100 are 561 wide tiles: up to three per workgroup.
# Steps of 128 columns: one; an odd number (a last chunk of one step); 17 and 33 (one block more than the 16 of a
# zero-point product, and than two of them); blocks of two and four steps; one block of three.
@pytest.mark.parametrize("m,n,k,c,bits,asym", [
    (1030, 2052, 128, 128, 4, True), (1030, 2052, 2176, 128, 4, True), (1030, 2052, 4224, 128, 4, True),
    (2050, 4100, 640, 128, 4, True), (1030, 2052, 640, 128, 4, False), (2050, 4100, 640, 128, 8, False),
    (1030, 2052, 2304, 256, 4, False), (1030, 2052, 1536, 512, 8, False), (1030, 2052, 384, -1, 4, False),
])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16])
def test_wide_tiles(ops, m, n, k, c, bits, asym, xdt):
  if c == -1:
    x, w, s, _ = cases.per_channel_int8(m, n, k, xdt, xdt, seed=m)
    w, z = w.clamp(-8, 7), None
  else:
    x, w, s, z, _ = cases.blockwise(m, n, k, c, bits, xdt, symmetric=not asym, seed=m + k)
    z = z if asym else None
  exp = oracle.quantized_matmul(x, w, s, z, block_size=c, int4_weight=bits == 4)
  before = ops.counters["wo_gemm"]
  out = torch.ops.xla.quantized_matmul(x.cuda(), w.cuda(), s.cuda(), None if z is None else z.cuda(), c, bits == 4).cpu()
  assert ops.counters["wo_gemm"] == before + 1
  # f32 sums in another order: a dot product rounds to its other neighbour now and then (the bound of the narrow tiles)
  assert cases.within_tolerance(out, exp)
  assert cases.rel_l2(out, exp) < 1e-3
  # an infinity stays in its row: rows of the same tile and lane group are untouched
  x[5, 3] = float("inf")
  bad = torch.ops.xla.quantized_matmul(x.cuda(), w.cuda(), s.cuda(), None if z is None else z.cuda(), c, bits == 4).cpu()
  keep = torch.arange(m) != 5
  assert torch.equal(bad[keep], out[keep])
  assert not torch.isfinite(bad[5]).any()
