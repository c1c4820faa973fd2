"""The matmuls against a row-major weight whose K is no multiple of the other kernels' steps, against the oracle."""
import numpy as np
import pytest
import torch

from oracle import quantized_matmul_oracle as oracle
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
  import xla_amd.experimental.custom_kernel  # noqa: F401
  import xla_amd.experimental.xla_quantized_matmul as m
  return m


# (m, n, k): one chunk of 64 columns less one, one more, whole chunks; row tiles of 16 / 32 / 64 with remainders; one
# column; fewer chunks than waves along K and more; channels per workgroup 16, 64 and 256
SHAPES = [(1, 1, 1), (3, 17, 63), (16, 16, 65), (17, 100, 192), (33, 31, 1000), (64, 130, 1030), (65, 70, 450),
          (1, 32777, 129), (300, 7000, 137), (1100, 8100, 67)]


@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("zp", [False, True])
def test_weight_only_any_k(ops, xdt, zp):
  for (m, n, k) in SHAPES:
    x, w, s, _ = cases.per_channel_int8(m, n, k, xdt, xdt, seed=m + n + k)
    z = (torch.randn(n, generator=cases.gen(5)) * 0.01).to(xdt) if zp else None
    exp = oracle.quantized_matmul(x, w, s, z)
    before = ops.counters["generic"]
    out = torch.ops.xla.quantized_matmul(x.cuda(), w.cuda(), s.cuda(), None if z is None else z.cuda()).cpu()
    assert ops.counters["generic"] == before + 1
    assert out.dtype == exp.dtype and out.shape == exp.shape
    assert cases.within_tolerance(out, exp), (m, n, k)
    if xdt == torch.float32:
      # sums of k products in two orders: at most about 2 sqrt(k) units of 2^-24 apart in the 2-norm (k <= 1030)
      assert cases.rel_l2(out, exp) < 4e-6, (m, n, k)


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (17, 33, 63), (64, 70, 130), (33, 5000, 1001), (1030, 8300, 71), (500, 4200, 72)])
def test_int8_product_any_k_exact(ops, m, n, k):
  g = cases.gen(m + n + k)
  xq = torch.randint(-128, 128, (m, k), generator=g, dtype=torch.int32).to(torch.int8)
  w = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int32).to(torch.int8)
  xs, ws = torch.rand(m, 1, generator=g), torch.rand(n, generator=g)
  zp, xsum = torch.randn(n, generator=g), xq.to(torch.int32).sum(-1)
  out, acc = ops.w8a8_gemm_gpu(xq.cuda(), w.cuda(), xs.cuda(), ws.cuda(), zp.cuda(), xsum.to(torch.int32).cuda(),
                               cvt_dtype=torch.float32, mid_dtype=torch.float32, out_dtype=torch.float32, want_acc=True)
  ref = torch.from_numpy(xq.numpy().astype(np.float64) @ w.numpy().astype(np.float64).T)  # (exact: below 2^53)
  assert torch.equal(acc.cpu().double(), ref)
  exp = (ref.float() * ws - xsum.float()[:, None] * zp) * xs
  torch.testing.assert_close(out.cpu(), exp, rtol=1e-6, atol=1e-2 * float(exp.abs().max()) * 1e-4)


# one row more than 65535 tiles of 16 rows, and than the 65535 tiles of 64 that one launch covers
@pytest.mark.parametrize("m", [65535 * 16 + 1, 65535 * 64 + 1])
def test_rows_past_one_grid(ops, m):
  k, n, last = 20, 3, 200
  g = cases.gen(m)
  x = torch.randn(last, k, generator=g).to(torch.bfloat16)
  w = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int32).to(torch.int8)
  s, z = torch.rand(n, generator=g).to(torch.bfloat16), torch.randn(n, generator=g).to(torch.bfloat16)
  xd = torch.zeros(m, k, dtype=torch.bfloat16, device="cuda")
  xd[-last:] = x.cuda()
  out = torch.ops.xla.quantized_matmul(xd, w.cuda(), s.cuda(), z.cuda())
  exp = oracle.quantized_matmul(x, w, s, z)
  assert cases.within_tolerance(out[-last:].cpu(), exp) and not out[:-last].any()
  # the int8 product: exact sums
  xq = torch.zeros(m, k, dtype=torch.int8, device="cuda")
  xq[-last:] = torch.randint(-128, 128, (last, k), generator=g, dtype=torch.int32).to(torch.int8).cuda()
  f32 = dict(cvt_dtype=torch.float32, mid_dtype=torch.float32, out_dtype=torch.float32)
  xs = torch.rand(m, 1, generator=g).cuda()
  out, acc = ops.w8a8_gemm_gpu(xq, w.cuda(), xs, s.float().cuda(), None, None, want_acc=True, **f32)
  want = xq[-last:].cpu().int() @ w.int().t()
  assert torch.equal(acc[-last:].cpu(), want) and not acc[:-last].any()
  assert torch.equal(out[-last:].cpu(), want.float() * s.float() * xs[-last:].cpu())


# one thread per output on either side of where it begins: by columns, by outputs (512 x 512), few rows against many
# channels; more outputs than the threads of its grid
SHORT = [(1, 1, 1), (7, 300, 16), (7, 300, 17), (7, 301, 47), (7, 301, 49), (301, 801, 31), (301, 801, 33), (512, 512, 15), (513, 512, 8), (513, 512, 9),
         (4, 32768, 40), (4, 32769, 41), (5, 32768, 9), (2100, 8200, 3)]


@pytest.mark.parametrize("m,n,k", SHORT)
def test_short_rows(ops, m, n, k):
  g = cases.gen(m + n + k)
  for xdt in (torch.bfloat16, torch.float16, torch.float32):
    x, w, s, _ = cases.per_channel_int8(m, n, k, xdt, xdt, seed=m + n + k)
    for z in (None, (torch.randn(n, generator=g) * 0.01).to(xdt)):
      exp = oracle.quantized_matmul(x, w, s, z)
      out = torch.ops.xla.quantized_matmul(x.cuda(), w.cuda(), s.cuda(), None if z is None else z.cuda()).cpu()
      assert out.dtype == exp.dtype and cases.within_tolerance(out, exp), (xdt, z is None)
  xq = torch.randint(-128, 128, (m, k), generator=g, dtype=torch.int32).to(torch.int8)
  xs, ws, zp = torch.rand(m, 1, generator=g), torch.rand(n, generator=g), torch.randn(n, generator=g)
  xsum = xq.to(torch.int32).sum(-1).to(torch.int32)
  f32 = dict(cvt_dtype=torch.float32, mid_dtype=torch.float32, out_dtype=torch.float32)
  out, acc = ops.w8a8_gemm_gpu(xq.cuda(), w.cuda(), xs.cuda(), ws.cuda(), zp.cuda(), xsum.cuda(), want_acc=True, **f32)
  ref = (xq.double() @ w.double().t()).float()  # (exact)
  assert torch.equal(acc.cpu().float(), ref)
  exp = (ref * ws - xsum.float()[:, None] * zp) * xs
  torch.testing.assert_close(out.cpu(), exp, rtol=1e-6, atol=1e-6 * float(exp.abs().max()))
