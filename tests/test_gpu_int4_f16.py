"""Int4 weights against f16 rows whose block sums lie at the ends of f16's range: rounded where the statement rounds them."""
import pytest
import torch

from tests import launch_recorder as rec

# (m, n, k, block, zero point, kernel): the streaming kernel, with eight half steps and over K slices; K split over waves;
# the 64 x 128 tiles with blocks of one step and of two, and with a single block (per channel); the 64 x 256 tiles
SHAPES = [
    (1, 64, 512, 128, True, "qmm_skinny_kernel"), (16, 256, 4096, 128, True, "qmm_skinny_kernel"),
    (12, 256, 8192, 128, False, "qmm_skinny_kernel"), (40, 132, 640, 128, True, "qmm_wo_bw_gemm_kernel_ksplit"),
    (260, 3000, 384, 128, True, "qmm_wo_bw_gemm_kernelI"), (300, 4096, 512, 256, False, "qmm_wo_bw_gemm_kernelI"),
    (130, 3000, 128, 128, False, "qmm_wo_bw_gemm_kernelI"), (1030, 2052, 256, 128, True, "qmm_wo_bw_wide_kernel"),
]


def test_kernels_of_the_shapes(tmp_path):
  f16 = 2
  calls = [(rec.skinny if m <= 16 and k < 8192 else rec.blockwise)(m, n, k, c, 4, zp, f16) for m, n, k, c, zp, _ in SHAPES]
  for shape, (rc, text, launches) in zip(SHAPES, rec.record(calls, str(tmp_path))):
    assert rc == 0 and shape[-1] in launches[0].name and len(launches) == (2 if shape[2] == 8192 else 1), (shape, text, launches)


def _spacing(v):
  """Distance of neighbouring f16 values at |v|."""
  return torch.exp2((v.abs().clamp(min=2.0**-14).log2().floor() - 10).clamp(max=6))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,c,zp,kernel", SHAPES)
def test_small_and_large_block_sums(m, n, k, c, zp, kernel):
  import xla_amd.experimental.custom_kernel  # noqa: F401
  g = torch.Generator().manual_seed(m + n)
  s = k // c
  # two weights of 1 or 2 per block; rows of about 1e-4 (block sums of 7e-5 .. 6e-4), the last one of +-16384 in turn
  # (sums of multiples of 16384: from 65536 on they are infinite; block sums of x are zero)
  w = torch.zeros(s, c, n, dtype=torch.int8)
  at = torch.rand(s, c, n, generator=g).topk(2, dim=1).indices
  w.scatter_(1, at, torch.randint(1, 3, (s, 2, n), generator=g, dtype=torch.int8) *
             (1 - 2 * torch.randint(0, 2, (s, 2, n), generator=g, dtype=torch.int8)))
  x = ((torch.rand(m, k, generator=g) * 0.7 + 0.7) * 1e-4 * (1 - 2 * torch.randint(0, 2, (m, k), generator=g))).half()
  if m > 1:
    x[m - 1] = 16384.0 * (1 - 2 * (torch.arange(k) % 2))
  scale = (torch.rand(s, n, generator=g) * 32 + 32).half()
  zero = (torch.rand(s, n, generator=g) * 0.25).half() if zp else None
  out = torch.ops.xla.quantized_matmul(x.cuda(), w.cuda(), scale.cuda(), None if zero is None else zero.cuda(), c, True)

  xb = x.double().reshape(m, s, c)
  dot = torch.matmul(xb.transpose(0, 1), w.double()).half().double()  # [s, m, n]
  exp = (scale.double()[:, None] * dot).sum(0)
  # a block's f32 sum of (16 + u) x less 24 sum x is off by some 2^-24 of what it adds up (0.25 at 128 columns), a spacing
  # of f16 at these sums (2^-24 - 2^-21): the rounded one is its neighbour, or the next.  In f16 sixteenths, rounded
  # before the factor, it would be off by up to eight of them.
  bound = (scale.double()[:, None] * 2 * _spacing(dot) * (c // 128)).sum(0)
  exp = exp.half().double()
  bound += _spacing(exp)
  if zp:
    xsum = xb.sum(2).half().double()  # [m, s]
    z = xsum @ zero.double()
    bound += _spacing(xsum) @ zero.double() + _spacing(z.half().double())
    exp = (exp - z.half().double()).half().double()
    bound += _spacing(exp)
  got = out.cpu().double()
  assert out.dtype == torch.float16
  fin = torch.isfinite(exp)
  assert torch.equal(torch.isfinite(got), fin) and torch.equal(torch.isnan(got), torch.isnan(exp))
  assert ((got - exp).abs()[fin] <= bound[fin]).all(), ((got - exp).abs() / bound)[fin].max()
  if m > 1:
    assert torch.equal(got[m - 1][~torch.isnan(exp[m - 1])], exp[m - 1][~torch.isnan(exp[m - 1])])
