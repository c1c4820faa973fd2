"""The last chunk of a row-major weight's rows, which begins before the row's whole chunks end, and tiles of 48 rows."""
import pytest
import torch

from oracle import quantized_matmul_oracle as oracle
from tests import cases

pytestmark = pytest.mark.gpu


# (m, n, k): rows of less than a chunk, a chunk, and one column less or more than some; a last chunk that is all but one
# column the one before it; 33 .. 48 rows (tiles of 48) with 16 and 64 channels per workgroup
SHAPES = [(1, 40, 63), (1, 40, 66), (17, 33, 65), (33, 100, 127), (40, 300, 130), (48, 70, 190), (48, 4100, 67), (49, 64, 571)]


@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("zp", [False, True])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_row_end(m, n, k, zp, xdt):
  import xla_amd.experimental.custom_kernel  # noqa: F401
  x, w, s, _ = cases.per_channel_int8(m, n, k, xdt, xdt, seed=m + n + k)
  z = (torch.randn(n, generator=cases.gen(5)) * 0.01).to(xdt) if zp else None
  args = [w.cuda(), s.cuda(), None if z is None else z.cuda()]
  out = torch.ops.xla.quantized_matmul(x.cuda(), *args).cpu()
  assert cases.within_tolerance(out, oracle.quantized_matmul(x, w, s, z))
  # an infinity in any column reaches its own row and no other one
  for col in (0, max(k - 64, 0), k // 64 * 64 - 1 if k > 64 else 0, k - 1):
    bad = x.clone()
    bad[m // 2, col] = float("inf")
    got = torch.ops.xla.quantized_matmul(bad.cuda(), *args).cpu()
    hit = w[:, col] != 0  # (0 * inf is NaN, or the zero point's infinity)
    assert not torch.isfinite(got[m // 2][hit]).any()
    rows = torch.arange(m) != m // 2
    assert torch.equal(got[rows], out[rows])
  ones = torch.ones(m, k, dtype=xdt)
  unit = torch.ones(n, dtype=xdt)
  # a column that two chunks hold is counted once: sums of 0s and 1s, exact in 32 bits and then rounded once to x's type
  few = (w.int() & 1).to(torch.int8)
  got = torch.ops.xla.quantized_matmul(ones.cuda(), few.cuda(), unit.cuda(), None).cpu()
  assert torch.equal(got, few.int().sum(1).to(torch.float32).to(xdt).expand(m, n))


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_row_end_int8_exact(m, n, k):
  import xla_amd.experimental.xla_quantized_matmul as ops
  g = cases.gen(m + n + k)
  xq, w = (torch.randint(-128, 128, (r, k), generator=g, dtype=torch.int32).to(torch.int8) for r in (m, n))
  one = torch.ones
  _, acc = ops.w8a8_gemm_gpu(xq.cuda(), w.cuda(), one(m, 1).cuda(), one(n).cuda(), None, None,
                             cvt_dtype=torch.float32, mid_dtype=torch.float32, out_dtype=torch.float32, want_acc=True)
  assert torch.equal(acc.cpu().double(), xq.double() @ w.double().t())  # (exact: below 2^53)
