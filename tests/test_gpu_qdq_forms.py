"""Quantize / dequantize per channel: every way the kernels address a tensor, against torch's own CPU operators."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def qd():
  import xla_amd.experimental.quantized  # noqa: F401  (binds the CUDA key)
  return torch.ops.quantized_decomposed


# axis 0, a run within a channel: rows of one run, of an odd number of runs, of no whole run (element by element; 4 and
# 12 are whole runs for an f32 result only); along the last axis: one to three groups of 8 rows with a remainder, a
# single run per row, channels of no whole run; in the middle; results past the size from which they are streamed and an
# input past it.
@pytest.mark.parametrize("shape,axis", [
    ((3, 8), 0), ((5, 4104), 0), ((7, 12), 0), ((9, 4), 0), ((5, 13), 0), ((1, 40960), 0),
    ((1, 8), 1), ((7, 8), 1), ((17, 4096), 1), ((24, 72), 1), ((9, 12), 1), ((9, 13), 1),
    ((3, 5, 16), 1), ((2, 3, 8), 2), ((4300, 4104), 0), ((4300, 4104), 1), ((8200, 8200), 0),
])
@pytest.mark.parametrize("scale_dtype,zp_dtype", [(torch.float32, torch.int64), (torch.bfloat16, torch.int32)])
def test_forms(qd, shape, axis, scale_dtype, zp_dtype):
  g = torch.Generator().manual_seed(sum(shape))
  big = shape[0] > 8000
  if big and scale_dtype != torch.float32:
    pytest.skip("once is enough")
  c = shape[axis]
  x = torch.randn(shape, generator=g) * 3
  x.view(-1)[1] = float("nan")
  x.view(-1)[2] = float("inf")
  scale = (torch.rand(c, generator=g) * 0.1 + 0.01).to(scale_dtype)
  zp = torch.randint(0, 100, (c,), generator=g).to(zp_dtype)
  for xdt in (torch.float32,) if big else (torch.float32, torch.bfloat16, torch.float16):
    for qdt, lo, hi in ((torch.int8, -128, 127), (torch.uint8, 0, 255)):
      xi = x.to(xdt)
      q = qd.quantize_per_channel(xi.cuda(), scale.cuda(), zp.cuda(), axis, lo, hi, qdt)
      want = qd.quantize_per_channel(xi.nan_to_num(nan=0.0, posinf=float("inf")).float(), scale.float(), zp, axis, lo, hi, qdt)
      got = q.cpu()
      same = got == want
      same.view(-1)[1] = got.view(-1)[1] == 0  # (NaN)
      assert same.all()
      for odt in (torch.float32, torch.bfloat16):
        d = qd.dequantize_per_channel(q, scale.cuda(), zp.cuda(), axis, lo, hi, qdt, out_dtype=odt)
        dw = qd.dequantize_per_channel(got, scale.float(), zp, axis, lo, hi, qdt).to(odt)
        assert d.dtype == odt and torch.equal(d.cpu(), dw)
