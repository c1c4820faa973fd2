"""W8A8: the tiles with three stages and two K groups, and the quantizer's thread counts, at their edges."""
import ctypes

import pytest
import torch

from xla_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
  import xla_amd.experimental.xla_quantized_matmul as q
  return q


def _int_operands(m, n, k):
  g = torch.Generator().manual_seed(m + n + k)
  x = torch.randint(-128, 128, (m, k), generator=g, dtype=torch.int8)
  w = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int8)
  return x, w, torch.rand(m, generator=g), torch.rand(n, generator=g)


def _check(ops, m, n, k, **kw):
  x, w, xs, ws = _int_operands(m, n, k)
  exact = x.double() @ w.double().t()  # (sums below 2^53)
  f32 = dict(cvt_dtype=torch.float32, mid_dtype=torch.float32, out_dtype=torch.float32)
  out, acc = ops.w8a8_gemm_gpu(x.cuda(), w.cuda(), xs.cuda(), ws.cuda(), None, None, want_acc=True, **f32, **kw)
  assert torch.equal(acc.cpu().double(), exact)
  want = (exact.float() * ws) * xs[:, None]
  assert torch.equal(out.cpu(), want)
  out, _ = ops.w8a8_gemm_gpu(x.cuda(), w.cuda(), xs.cuda(), ws.cuda(), None, None, **f32, **kw)  # the short epilogue
  assert torch.equal(out.cpu(), want)


# 128 x 256 tiles: one to five K steps (three stages: two are copied ahead), a partial last step, row and column tails
@pytest.mark.parametrize("k", [128, 256, 272, 384, 640, 1040])
@pytest.mark.parametrize("m,n", [(128, 256), (300, 600), (129, 258)])
def test_128x256(ops, m, n, k):
  _check(ops, m, n, k, block_m=128, block_n=256)


# more than 256 tiles of 64 x 64, at most 256 of 64 x 128, K from 4096, more than two row tiles (else 64 x 64): an even and an odd number of steps, a partial one
@pytest.mark.parametrize("m,n,k", [(130, 5512, 4096), (130, 5511, 4112), (200, 4228, 4224), (33, 16500, 4096),
                                   (129, 5500, 4096)])
def test_64x128_two_k_groups(ops, m, n, k):
  tile = (ctypes.c_int32 * 3)()
  assert _lib.load().xla_amd_qmm_w8a8_tile(m, n, k, tile) == 0 and tuple(tile)[:2] == (64, 128 if m > 128 else 64)
  _check(ops, m, n, k)


# asked for at any size: fewer steps of K than the two groups, one each, more; row and column tails
@pytest.mark.parametrize("m,n,k", [(64, 128, 16), (65, 129, 128), (30, 100, 144), (100, 300, 256), (1, 1, 1040)])
def test_64x128_asked_for(ops, m, n, k):
  _check(ops, m, n, k, block_m=64, block_n=128)


# 128 x 128 tiles: three stages with one tile per compute unit at most, two with more
@pytest.mark.parametrize("m,n,k", [(128, 128, 128), (129, 258, 272), (300, 200, 1040), (2100, 2100, 400)])
def test_128x128_asked_for(ops, m, n, k):
  _check(ops, m, n, k, block_m=128, block_n=128)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_quantizer_thread_counts(ops, dtype):
  for k in (2048, 2056, 4096, 4104, 8192, 8200, 16384, 16392):
    for m in (1, 256, 257):
      x = (torch.randn(m, k, generator=torch.Generator().manual_seed(k + m)) * 3).to(dtype)
      x[0, k - 1] = 50.0  # the maximum in the last thread's share
      q, s, xsum = ops.quantize_per_token_gpu(x.cuda(), want_sum=True)
      qw, sw = ops._quantize_tensor(x)
      assert torch.equal(q.cpu(), qw) and torch.equal(s.cpu(), sw), (dtype, m, k)
      assert torch.equal(xsum.cpu(), qw.int().sum(-1, dtype=torch.int32))


# many rows of up to 6144 (f32: 4096) elements take 256 threads: either side of where
@pytest.mark.parametrize("dtype,k,rows", [(torch.bfloat16, 4104, (767, 768)), (torch.float16, 6144, (768,)), (torch.bfloat16, 6152, (768,)),
                                          (torch.float32, 2056, (1535, 1536)), (torch.float32, 4096, (1536,))])
def test_quantizer_many_rows(ops, dtype, k, rows):
  for m in rows:
    x = (torch.randn(m, k, generator=torch.Generator().manual_seed(k + m)) * 3).to(dtype)
    x[0, k - 1], x[m - 1, 0] = 50.0, -60.0
    q, s, xsum = ops.quantize_per_token_gpu(x.cuda(), want_sum=True)
    qw, sw = ops._quantize_tensor(x)
    assert torch.equal(q.cpu(), qw) and torch.equal(s.cpu(), sw)
    assert torch.equal(xsum.cpu(), qw.int().sum(-1, dtype=torch.int32))
