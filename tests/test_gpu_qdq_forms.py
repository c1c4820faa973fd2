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


@pytest.mark.parametrize("shape", [(1, 1, 24), (1, 3, 8), (1, 8, 1), (1, 72, 1), (7, 8, 1), (9, 24, 1), (5, 13, 1),
                                   (2, 131080, 1), (33, 8192, 1)])
def test_nothing_past_the_end(shape):
  """Tensors of less than a workgroup, and rows that do not fill their last group: the results end where they should (threads that have no elements write none)."""
  from xla_amd import _lib
  lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
  o, c, i = shape
  n, room = o * c * i, max(1 << 14, 2 * o * c * i)
  scale, zp = torch.rand(c, device="cuda") + 0.5, torch.randint(-5, 5, (c,), dtype=torch.int32, device="cuda")
  x = torch.randn(room, device="cuda") * 50
  q = torch.full((room,), 77, dtype=torch.int8, device="cuda")
  _lib.check(lib.xla_amd_qmm_quantize_affine(x.data_ptr(), q.data_ptr(), scale.data_ptr(), zp.data_ptr(), o, c, i,
                                             _lib.DT_F32, _lib.QDT_I8, -128, 127, stream), "quantize")
  assert (q[n:] == 77).all()
  s, z = scale.view(1, c, 1), zp.view(1, c, 1)
  want = ((x[:n].view(o, c, i) * s).round() + z).clamp(-128, 127)
  assert torch.equal(q[:n].view(o, c, i).float(), want)
  for dtype in (torch.float32, torch.bfloat16, torch.float16):
    out = torch.full((room,), -7.0, dtype=dtype, device="cuda")
    _lib.check(lib.xla_amd_qmm_dequantize_affine(q.data_ptr(), out.data_ptr(), scale.data_ptr(), zp.data_ptr(), o, c, i,
                                                 _lib.QDT_I8, _lib.dt(dtype), 1, stream), "dequantize")
    assert (out[n:] == -7).all()
    assert torch.equal(out[:n].view(o, c, i), ((want - z) * s).to(dtype))


# along the last axis from the size on at which a thread takes eight channels of several rows: a single run per row, two
# rows, an odd row past whole groups, channels of no whole run
@pytest.mark.parametrize("shape,axis", [((32768, 8), 1), ((2, 131072), 1), ((65, 4096), 1), ((33, 8200), 1), ((4100, 5, 16), 2), ((2100, 129), 1)])
@pytest.mark.parametrize("scale_dtype,zp_dtype", [(torch.float32, torch.int64), (torch.float16, torch.int32)])
def test_several_rows_along_the_last_axis(qd, shape, axis, scale_dtype, zp_dtype):
  test_forms(qd, shape, axis, scale_dtype, zp_dtype)


def test_parameters_at_any_element(qd):
  """Scales and zero points that are slices of longer tensors start at any element's address."""
  g = torch.Generator().manual_seed(3)
  x = (torch.randn(64, 8192, generator=g) * 3).cuda()
  scale, zp = (torch.rand(8200, generator=g) * 0.1 + 0.01).cuda(), torch.randint(0, 100, (8200,), generator=g).cuda()
  for sdt in (torch.float32, torch.bfloat16):
    for zdt in (torch.int64, torch.int32):
      s, z = scale.to(sdt)[3:8195], zp.to(zdt)[5:8197]
      q = qd.quantize_per_channel(x, s, z, 1, -128, 127, torch.int8)
      assert torch.equal(q, qd.quantize_per_channel(x, s.clone(), z.clone(), 1, -128, 127, torch.int8))
      want = qd.quantize_per_channel(x.cpu(), s.float().cpu(), z.cpu(), 1, -128, 127, torch.int8)
      assert torch.equal(q.cpu(), want)
