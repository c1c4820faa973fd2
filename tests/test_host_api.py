"""Host-side checks that need no GPU: the C-ABI library loads and exports what
include/xla_amd_qmm.h declares, the dispatcher, operator registration, argument
checks with the reference's messages, the module and the quantizer utilities."""
import ctypes
import os
import re
import subprocess
import sys

import pytest
import torch

from oracle import quantized_matmul_oracle as oracle
from tests import cases
from xla_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def qmm():
  import xla_amd.experimental.custom_kernel  # noqa: F401
  import xla_amd.experimental.xla_quantized_matmul as m
  return m


def declared_functions():
  text = open(os.path.join(ROOT, "include", "xla_amd_qmm.h")).read()
  text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
  return sorted(set(re.findall(r"\b(xla_amd_qmm_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
  lib = _lib.load()
  names = declared_functions()
  assert len(names) >= 10
  for n in names:
    assert hasattr(lib, n), f"{n} declared in the header but not exported"
  assert sorted(_lib.SIGNATURES) == names, "ctypes signatures out of sync with the header"
  assert lib.xla_amd_qmm_abi_version() == 5


def test_header_cites_reference_for_each_entry_point():
  text = open(os.path.join(ROOT, "include", "xla_amd_qmm.h")).read()
  for key in ("xla_quantized_matmul.py", "custom_kernel.py", "dot_general.cpp", "cast_int4.cpp",
              "quantized_matmul_kernel.py"):
    assert key in text


def test_dispatcher_regimes():
  lib = _lib.load()
  d = lib.xla_amd_qmm_dispatch
  assert d(16, 14336, 4096, 4096, 8, _lib.DT_BF16, 0) == _lib.KERNEL_SKINNY_MFMA
  assert d(1, 4096, 4096, 128, 4, _lib.DT_BF16, 0) == _lib.KERNEL_SKINNY_MFMA
  assert d(3, 8, 5, 5, 8, _lib.DT_F32, 0) == _lib.KERNEL_GENERIC
  assert d(3, 8, 6, 2, 8, _lib.DT_F32, 0) == _lib.KERNEL_GENERIC
  # weight-only, per-channel int8, 2-byte x: more than 32 rows take the tiled GEMM; so do few rows against few
  # channels and a long K (the streaming kernel over K slices, behind the same entry point with a workspace)
  assert d(33, 14336, 4096, 4096, 8, _lib.DT_BF16, 0) == _lib.KERNEL_WEIGHT_ONLY_GEMM
  assert d(2048, 14336, 4096, 4096, 8, _lib.DT_F16, 0) == _lib.KERNEL_WEIGHT_ONLY_GEMM
  assert d(2048, 14336, 4096, 4096, 8, _lib.DT_F32, 0) == _lib.KERNEL_WEIGHT_ONLY_GEMM  # f32 rows, split into bf16 parts
  assert d(127, 14336, 4096, 4096, 8, _lib.DT_F32, 0) == _lib.KERNEL_SKINNY_MFMA         # fewer than 128: 16 per pass
  assert d(128, 14336, 4096, 4096, 8, _lib.DT_F32, 0) == _lib.KERNEL_WEIGHT_ONLY_GEMM
  assert d(2048, 14336, 4096 + 64, 4096 + 64, 8, _lib.DT_F32, 0) == _lib.KERNEL_GENERIC
  assert lib.xla_amd_qmm_weight_only_gemm_f32_workspace_bytes(2048, 14336, 4096) == 2048 * 4096 * 6
  assert lib.xla_amd_qmm_weight_only_gemm_f32_workspace_bytes(2048, 14336, 4100) == 0
  assert d(2048, 4096, 4096, 128, 8, _lib.DT_BF16, 0) == _lib.KERNEL_WEIGHT_ONLY_GEMM  # blockwise: its own tiled GEMM
  assert d(2048, 14336, 4096, 4096, 4, _lib.DT_BF16, 0) == _lib.KERNEL_WEIGHT_ONLY_GEMM  # int4 too
  assert d(64, 4096, 4096, 128, 4, _lib.DT_BF16, 0) == _lib.KERNEL_SKINNY_MFMA         # up to 64 rows stream (two passes)
  assert d(2048, 4096, 4096, 128, 4, _lib.DT_F32, 0) == _lib.KERNEL_SKINNY_MFMA        # f32 x: no GEMM
  assert d(100, 30, 256, 128, 8, _lib.DT_BF16, 0) == _lib.KERNEL_GENERIC               # blockwise needs N % 4 == 0
  assert lib.xla_amd_qmm_weight_only_gemm_workspace_bytes(2048, 4096, 4096, 128, 4) == 0
  assert d(32, 4096, 14336, 14336, 4, _lib.DT_BF16, 0) == _lib.KERNEL_WEIGHT_ONLY_GEMM  # int4 K slices (steps of 1024 columns)
  assert lib.xla_amd_qmm_weight_only_gemm_workspace_bytes(32, 4096, 14336, 14336, 4) == 4 * (32 * 4096 + 32) * 4
  assert d(32, 4096, 14336, 128, 4, _lib.DT_BF16, 0) == _lib.KERNEL_WEIGHT_ONLY_GEMM     # blockwise K slices (whole blocks)
  assert lib.xla_amd_qmm_weight_only_gemm_workspace_bytes(32, 4096, 14336, 128, 4) == 2 * 4 * 32 * 4096 * 4  # sums + zero-point sums
  assert d(32, 4096, 14336, 7168, 8, _lib.DT_BF16, 0) == _lib.KERNEL_SKINNY_MFMA         # a slice is whole blocks, at least two of them: two blocks stay one slice
  assert d(32, 4098, 14336, 128, 4, _lib.DT_BF16, 0) == _lib.KERNEL_GENERIC              # blockwise needs N % 4 == 0
  assert lib.xla_amd_qmm_weight_only_gemm_workspace_bytes(32, 4096, 14336, 2048, 8) == 2 * 3 * 32 * 4096 * 4  # 3 + 3 + 1 blocks
  assert d(32, 4096, 14336, 14336, 8, _lib.DT_BF16, 0) == _lib.KERNEL_WEIGHT_ONLY_GEMM
  assert d(4, 4096, 14336, 14336, 8, _lib.DT_BF16, 0) == _lib.KERNEL_SKINNY_MFMA      # too few rows of x to matter
  assert d(32, 4096, 4096, 4096, 8, _lib.DT_BF16, 0) == _lib.KERNEL_SKINNY_MFMA       # K too short for slices
  assert d(32, 1024, 4096, 4096, 8, _lib.DT_BF16, 0) == _lib.KERNEL_WEIGHT_ONLY_GEMM  # ... unless the output is narrow and x two tiles high
  assert d(16, 1024, 4096, 4096, 8, _lib.DT_BF16, 0) == _lib.KERNEL_SKINNY_MFMA
  assert d(32, 14336, 8192, 8192, 8, _lib.DT_BF16, 0) == _lib.KERNEL_SKINNY_MFMA      # enough workgroups already
  assert lib.xla_amd_qmm_weight_only_gemm_workspace_bytes(32, 4096, 14336, 14336, 8) == 4 * (32 * 4096 + 32) * 4  # four K slices
  assert lib.xla_amd_qmm_weight_only_gemm_workspace_bytes(2048, 14336, 4096, 4096, 8) == 0
  assert d(2048, 14336, 4096, 4096, 8, _lib.DT_BF16, 1) == _lib.KERNEL_W8A8_MFMA
  assert d(3, 8, 5, 5, 8, _lib.DT_F32, 1) == _lib.KERNEL_W8A8_GENERIC
  tile = (ctypes.c_int32 * 3)()
  assert lib.xla_amd_qmm_w8a8_tile(2048, 14336, 4096, tile) == 0
  assert list(tile) == [256, 256, 128]
  assert lib.xla_amd_qmm_w8a8_tile(64, 64, 64, tile) == 0 and list(tile)[:2] == [32, 32]  # few tiles: the smallest ones
  assert lib.xla_amd_qmm_w8a8_tile(128, 4096, 4096, tile) == 0 and list(tile)[:2] == [64, 32]  # 512 tiles of 32 x 32 would be two per CU
  assert lib.xla_amd_qmm_w8a8_tile(32, 4096, 14336, tile) == 0 and list(tile)[:2] == [32, 32]
  assert lib.xla_amd_qmm_w8a8_tile(128, 14336, 4096, tile) == 0 and list(tile)[:2] == [64, 64]
  # the shape-based choice agrees with the measured best of the tuning sweep on the Llama-3-8B prefill shapes
  from xla_amd.experimental.hip_kernels.quantized_matmul_kernel import TUNED_BLOCK_SIZES
  for (m, n, k) in [(2048, 6144, 4096), (2048, 4096, 4096), (1024, 4096, 4096), (512, 4096, 4096), (512, 14336, 4096),
                    (4096, 4096, 14336), (2048, 4096, 14336), (256, 28672, 4096), (8192, 1024, 4096), (32, 4096, 14336),
                    (64, 4096, 4096), (128, 4096, 14336), (512, 1024, 4096), (128, 6144, 4096), (256, 14336, 4096),
                    (128, 28672, 4096), (512, 6144, 4096)]:
    assert lib.xla_amd_qmm_w8a8_tile(m, n, k, tile) == 0
    assert tuple(tile) == TUNED_BLOCK_SIZES[("gfx950", m, n, k, "bfloat16", True)], (m, n, k)


def test_error_codes_without_gpu():
  lib = _lib.load()
  assert lib.xla_amd_qmm_packed_bytes(8, 64, 8) == 512
  assert lib.xla_amd_qmm_packed_bytes(8, 64, 4) == 256
  assert lib.xla_amd_qmm_packed_bytes(8, 5, 4) == 0
  assert lib.xla_amd_qmm_tiled_bytes(17, 256, 256, 8) == 32 * 256
  assert lib.xla_amd_qmm_tiled_bytes(16, 128, 128, 4) == 16 * 64
  assert lib.xla_amd_qmm_tiled_bytes(16, 64, 64, 8) == 0
  # channel groups of the tiled copy: 16, narrower where that fills the 1024 wave slots of the chip better
  # (per-channel int8 weights of 4096 channels or more only)
  group = lib.xla_amd_qmm_tile_group
  assert [group(n, 4096, 4096, 8) for n in (1024, 4096, 5120, 6144, 8192, 11008, 14336, 16384, 28672, 128256)] == \
      [16, 16, 10, 12, 16, 12, 14, 16, 14, 16]
  assert group(14336, 4096, 4096, 4) == 16 and group(14336, 4096, 128, 8) == 16 and group(14336, 4096, -1, 8) == 14
  assert lib.xla_amd_qmm_tiled_bytes(14336, 4096, 4096, 8) == 14336 * 4096          # 1024 groups of 14
  assert lib.xla_amd_qmm_tiled_bytes(7165, 256, 256, 8) == 512 * 14 * 256            # groups of 14, three channels of padding
  assert lib.xla_amd_qmm_tiled_bytes(7165, 256, 128, 8) == 448 * 16 * 256            # blockwise: groups of 16
  rc = lib.xla_amd_qmm_weight_only_skinny(None, None, None, None, None, 1, 1, 128, 128, 8, 1, 1, 1, 1, 1, 1, None)
  assert rc == _lib.EINVAL and b"null" in lib.xla_amd_qmm_last_error()
  rc = lib.xla_amd_qmm_quantize_per_token(None, None, None, None, 1, 1, 0, 0, 0, None)
  assert rc == _lib.EINVAL
  rc = lib.xla_amd_qmm_w8a8_gemm(None, None, None, None, None, None, None, None, 1, 1, 16, 0, 0, 0, 0, 0, 0, 0, 0, 0, None)
  assert rc == _lib.EINVAL
  with pytest.raises(RuntimeError, match="failed"):
    _lib.check(rc, "w8a8_gemm")
  assert lib.xla_amd_qmm_w8a8_linear_workspace_bytes(2048, 14336, 4096) >= 2048 * 4096 + 2 * 2048 * 4
  assert lib.xla_amd_qmm_w8a8_linear_workspace_bytes(3, 8, 5) % 256 == 0
  rc = lib.xla_amd_qmm_w8a8_linear(None, None, None, None, None, None, 0, 1, 1, 16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, None)
  assert rc == _lib.EINVAL and b"null" in lib.xla_amd_qmm_last_error()
  rc = lib.xla_amd_qmm_untile_weight(None, None, 1, 128, 16, 0, 8, None)
  assert rc == _lib.EINVAL


def test_ops_are_registered_with_reference_schemas(qmm):
  s = str(torch.ops.xla.quantized_matmul.default._schema)
  assert s == ("xla::quantized_matmul(Tensor x, Tensor w, Tensor scale, Tensor? zero_point=None, int? block_size=-1, "
               "bool? int4_weight=False, bool? quantize_activation=False) -> Tensor")
  s8 = str(torch.ops.xla.quantized_matmul_int8.default._schema)
  assert s8.startswith("xla::quantized_matmul_int8(Tensor x, Tensor w, Tensor scalar, Tensor? zero_point=None, "
                       "Tensor? quant_block_size=None, bool quantize_activation=False, int? batch_block_size=None")


def _gold():
  import json
  return json.load(open(os.path.join(ROOT, "tests", "golden", "quantized_matmul_golden.json")))


def _bf16_from_bits(bits):
  import numpy as np
  return torch.tensor(np.asarray(bits, dtype=np.uint16).astype(np.int32)).to(torch.int16).view(torch.bfloat16)


def test_cpu_tensors_against_fixtures_and_the_exact_model(qmm):
  # the CPU key is checked against data that shares no code with it: the hand-worked fixtures, the exact
  # integer / float64 model, and the reference's fake-quant identity
  import numpy as np
  from oracle import bitexact_model as bx
  op = torch.ops.xla.quantized_matmul
  g = _gold()["hand_per_channel"]
  x, w = torch.tensor(g["x"]), torch.tensor(g["w"], dtype=torch.int8)
  s, z = torch.tensor(g["scale"]), torch.tensor(g["zp"])
  assert torch.equal(op(x, w, s), torch.tensor(g["expect"]))
  assert torch.equal(op(x, w, s, z), torch.tensor(g["expect_zp"]))
  g = _gold()["hand_blockwise"]
  x, w = torch.tensor(g["x"]), torch.tensor(g["w"], dtype=torch.int8)
  s, z = torch.tensor(g["scale"]), torch.tensor(g["zp"])
  assert torch.equal(op(x, w, s, block_size=2), torch.tensor(g["expect"]))
  assert torch.equal(op(x, w, s, z, block_size=2), torch.tensor(g["expect_zp"]))
  # W8A8: quantizer and accumulators from the exact model, epilogue as written in the operator's contract
  x = cases.outlier_activations(32, 512, torch.bfloat16, seed=7)
  _, w, s, _ = cases.per_channel_int8(1, 48, 512, torch.bfloat16, torch.float32, seed=8)
  q, xs, _ = bx.quantize_rows(x.double().numpy(), "bf16", "saturate")
  acc = torch.tensor(bx.int_matmul(q, w.numpy()))
  expect = (acc.float() * s) * torch.tensor(xs, dtype=torch.float32)[:, None]
  out = op(x, w, s, quantize_activation=True)
  assert out.dtype == torch.float32 and torch.equal(out, expect)
  zp = torch.randn(48, generator=cases.gen(9)) * 0.01
  xsum = torch.tensor(q.sum(-1), dtype=torch.float32)[:, None]
  expect_zp = (acc.float() * s - xsum * zp) * torch.tensor(xs, dtype=torch.float32)[:, None]
  assert torch.equal(op(x, w, s, zp, quantize_activation=True), expect_zp)
  # blockwise asymmetric: x @ (w * scale - zp) in float64 (test_quantized_matmul.py:210-218)
  xb, wb, sb, zb, _ = cases.blockwise(6, 24, 64, 16, 4, torch.float32, symmetric=False, seed=2)
  ref = bx.dense_fake_quant(xb.numpy(), wb.permute(2, 0, 1).reshape(24, 64).numpy(), sb.numpy(), zb.numpy(), 16)
  assert np.abs(op(xb, wb, sb, zb, block_size=16).double().numpy() - ref).max() < 1e-5
  # bf16 weight-only: dot rounded to bf16, then scaled and rounded again
  x, w, s, _ = cases.per_channel_int8(16, 256, 1024, torch.bfloat16, torch.bfloat16, seed=6)
  two = ((x.double() @ w.double().T).to(torch.bfloat16).float() * s.float()).to(torch.bfloat16)
  out = op(x, w, s)
  assert out.dtype == torch.bfloat16 and cases.rel_l2(out, two) < 3e-4
  # batch dimensions, and agreement with the restatement of the reference's op sequence within tolerance
  x3 = torch.randn(2, 3, 64, generator=cases.gen(3))
  assert op(x3, wb, sb, zb, block_size=16).shape == (2, 3, 24)
  assert cases.within_tolerance(op(x3, wb, sb, zb, block_size=16), oracle.quantized_matmul(x3, wb, sb, zb, block_size=16))


def test_cpu_key_follows_the_overflow_policy(qmm, monkeypatch):
  # one operator, one answer: CPU tensors apply the float -> int8 policy of the GPU kernels
  g = _gold()["bf16_overflow_band"]
  x = _bf16_from_bits(g["maxima_bits"]).reshape(-1, 1)
  ident = torch.ones(1, 1, dtype=torch.int8)
  one = torch.ones(1)
  for policy in ("saturate", "wrap"):
    monkeypatch.setenv("XLA_AMD_QMM_OVERFLOW", policy)
    q, s = qmm._quantize_tensor(x)
    assert q.flatten().tolist() == g["q_" + policy]
    assert torch.equal(s.flatten(), _bf16_from_bits(g["scale_bits"]))
    # through the operator: out = q * 1 * x_scale
    out = torch.ops.xla.quantized_matmul(x, ident, one, quantize_activation=True)
    assert torch.equal(out.flatten(), torch.tensor(g["q_" + policy], dtype=torch.float32) * s.flatten().float())
  monkeypatch.delenv("XLA_AMD_QMM_OVERFLOW")
  assert qmm._overflow_policy() == "saturate"
  q, _ = qmm._quantize_tensor(x)
  assert q.flatten().tolist() == g["q_saturate"]
  z, zs = qmm._quantize_tensor(torch.zeros(2, 8, dtype=torch.bfloat16))
  assert z.abs().sum() == 0 and zs.abs().sum() == 0
  n, ns = qmm._quantize_tensor(torch.tensor([[1.0, float("nan"), 2.0]]))
  assert n.abs().sum() == 0 and torch.isnan(ns).all()


def test_meta_tensors(qmm):
  x = torch.empty(2, 3, 64, device="meta", dtype=torch.bfloat16)
  w = torch.empty(32, 64, device="meta", dtype=torch.int8)
  s = torch.empty(32, device="meta", dtype=torch.float32)
  assert torch.ops.xla.quantized_matmul(x, w, s).shape == (2, 3, 32)
  assert torch.ops.xla.quantized_matmul(x, w, s).dtype == torch.float32
  assert torch.ops.xla.quantized_matmul(x, w, s.bfloat16(), quantize_activation=True).dtype == torch.bfloat16
  x2 = torch.empty(10, 20, device="meta", dtype=torch.bfloat16)
  w2 = torch.empty(30, 20, device="meta", dtype=torch.int8)
  r = torch.ops.xla.quantized_matmul_int8(x2, w2, torch.empty(30, device="meta"), quantize_activation=True)
  assert r.shape == (10, 30) and r.dtype == torch.bfloat16  # test/test_pallas.py:1030-1045


def test_argument_checks_use_the_reference_messages(qmm):
  x = torch.randn(3, 5)
  w = torch.randint(-8, 8, (8, 5), dtype=torch.int8)
  s = torch.rand(8)
  with pytest.raises(AssertionError, match="Weight dtype is expected to be torch.int8"):
    torch.ops.xla.quantized_matmul(x, w.float(), s)
  with pytest.raises(AssertionError, match=r"Weight shape is expected to be \[output_dim, input_dim\]"):
    torch.ops.xla.quantized_matmul(torch.randn(3, 6), w, s)
  with pytest.raises(AssertionError, match="weight scaler shape is expect to be"):
    torch.ops.xla.quantized_matmul(x, w, torch.rand(8, 1))
  wb = torch.randint(-8, 8, (3, 2, 8), dtype=torch.int8)
  with pytest.raises(AssertionError, match="Blockwise quantization does not support activation quantization"):
    torch.ops.xla.quantized_matmul(torch.randn(3, 6), wb, torch.rand(3, 8), block_size=2, quantize_activation=True)
  with pytest.raises(AssertionError, match="Weight tensor is expected to be 3D"):
    torch.ops.xla.quantized_matmul(torch.randn(3, 6), torch.zeros(8, 6, dtype=torch.int8), torch.rand(3, 8), block_size=2)
  with pytest.raises(AssertionError, match="input_dim should be divisible by block_size"):
    torch.ops.xla.quantized_matmul(torch.randn(3, 7), wb, torch.rand(3, 8), block_size=2)


def test_module_matches_reference_layout(qmm):
  m = qmm.XlaQuantizedLinear(6, 8)
  assert sorted(m.state_dict()) == ["weight", "weight_scaler", "zero_point"]
  assert m.weight.dtype == torch.int8 and tuple(m.weight.shape) == (8, 6)
  assert sorted(qmm.XlaQuantizedLinear(6, 8, is_symmetric=True).state_dict()) == ["weight", "weight_scaler"]
  mb = qmm.XlaQuantizedLinear(6, 8, block_size=2)
  assert tuple(mb.weight.shape) == (8, 6)  # 2-D until load_quantized_weight swaps it (as in the reference)
  wb = torch.randint(-8, 8, (3, 2, 8), dtype=torch.int8)
  mb.load_quantized_weight(wb, torch.rand(3, 8), torch.rand(3, 8))
  assert tuple(mb.weight.shape) == (3, 2, 8)
  with pytest.raises(AssertionError):
    mb.load_quantized_weight(torch.zeros(8, 6, dtype=torch.int8), torch.rand(3, 8))
  x = torch.randn(4, 6)
  assert torch.allclose(mb(x), oracle.quantized_matmul(x, mb.weight, mb.weight_scaler, mb.zero_point, block_size=2), atol=1e-6)


def test_rtn_quantizer_and_module_swap(qmm):
  from xla_amd.quantization import quantize_weight_rtn, replace_linear_with_quantized
  g = cases.gen(5)
  w_fp = torch.randn(16, 64, generator=g) * 0.02
  for bits, block, sym in [(8, -1, True), (8, -1, False), (4, 16, False), (4, 16, True), (8, 32, False)]:
    w, s, z = quantize_weight_rtn(w_fp, bits, block, sym)
    qmin, qmax = -2**(bits - 1), 2**(bits - 1) - 1
    assert w.dtype == torch.int8 and w.min() >= qmin and w.max() <= qmax
    if block == -1:
      assert tuple(w.shape) == (16, 64) and tuple(s.shape) == (16,)
      deq = w.float() * s[:, None] - (0 if z is None else z[:, None])
    else:
      assert tuple(w.shape) == (64 // block, block, 16) and tuple(s.shape) == (64 // block, 16)
      deq = (w.float() * s[:, None, :] - (0 if z is None else z[:, None, :])).reshape(64, 16).T
    assert (deq - w_fp).abs().max() <= s.max() * 0.5 + 1e-6  # RTN error is at most half a step
  net = torch.nn.Sequential(torch.nn.Linear(64, 32, bias=False), torch.nn.ReLU(), torch.nn.Linear(32, 8, bias=True))
  x = torch.randn(5, 64, generator=g)
  ref = net(x)
  replace_linear_with_quantized(net, n_bits=8)
  assert isinstance(net[0], qmm.XlaQuantizedLinear) and isinstance(net[2], torch.nn.Linear)
  assert torch.allclose(net(x), ref, atol=0.05)


def _linear_model(n_in, n_out):
  class M(torch.nn.Module):
    def __init__(self):
      super().__init__()
      self.linear = torch.nn.Linear(n_in, n_out, bias=False)

    def forward(self, x):
      return self.linear(x)
  return M()


@pytest.mark.parametrize("quantize_activation", [False, True])
def test_q_linear_module_compile(qmm, quantize_activation):
  # test_quantized_matmul.py:128-143 (test_q_linear_module_dynamo) with the backends present here: the op has a
  # Meta implementation, so the module traces as one opaque call, without graph breaks
  from xla_amd.quantization import replace_linear_with_quantized
  torch.manual_seed(0)
  with torch.no_grad():
    m = _linear_model(5, 8)
    x = torch.randn(3, 5)
    out_fp = m(x)
    replace_linear_with_quantized(m, n_bits=8, quantize_activation=quantize_activation)
    out_quant = m(x)
    assert torch.allclose(out_fp, out_quant, atol=0.02)
    for backend in ("eager", "aot_eager"):
      torch._dynamo.reset()
      out_compiled = torch.compile(m, backend=backend, fullgraph=True)(x)
      assert torch.allclose(out_compiled, out_quant, atol=4e-3), backend


def test_tuned_block_table(qmm):
  from xla_amd.experimental.hip_kernels.quantized_matmul_kernel import TUNED_BLOCK_SIZES, get_tuned_block_sizes
  key0 = next(iter(TUNED_BLOCK_SIZES))
  arch, bs, n_out, n_in, dt, qa = key0
  assert get_tuned_block_sizes(TUNED_BLOCK_SIZES, bs, n_out, n_in, dt, qa, arch=arch) == TUNED_BLOCK_SIZES[key0]
  assert get_tuned_block_sizes(TUNED_BLOCK_SIZES, 7, 9, 11, "bfloat16", True, arch=arch) == (None, None, None)
  assert TUNED_BLOCK_SIZES[("gfx950", 2048, 14336, 4096, "bfloat16", True)] == (256, 256, 128)


def test_product_does_not_import_the_oracle():
  for dirpath, _, files in os.walk(os.path.join(ROOT, "xla_amd")):
    for f in files:
      if f.endswith((".py", ".hip", ".h", ".cpp")):
        text = open(os.path.join(dirpath, f)).read()
        assert "oracle" not in text.lower().replace("no fallback", ""), f"{f} mentions the oracle"


def test_fuse_quantized_linears_cpu():
  # N-concatenated layers give the outputs of the separate layers (CPU operator path; to the last bits only: the
  # host's matrix multiply may block a 48-column product differently from a 24-column one)
  import xla_amd.experimental.custom_kernel  # noqa: F401
  from xla_amd.quantization import quantize_linear, fuse_quantized_linears
  torch.manual_seed(3)
  x = torch.randn(5, 64)
  for kwargs in (dict(n_bits=8), dict(n_bits=8, symmetric=False), dict(n_bits=4, block_size=32, symmetric=False)):
    lins = [quantize_linear(torch.nn.Linear(64, n, bias=False), **kwargs) for n in (24, 8, 16)]
    fused = fuse_quantized_linears(lins)
    outs = fused(x).split([l.output_dim for l in lins], dim=-1)
    for l, o in zip(lins, outs):
      torch.testing.assert_close(l(x), o, rtol=1e-5, atol=1e-6, msg=str(kwargs))


def test_no_kernel_of_the_built_library_spills_registers():
  """The build writes every kernel's resources; a scratch frame (register spills) is a silent slowdown of several times."""
  import json
  from xla_amd import build
  if not os.path.exists(build.RESOURCES_PATH):
    pytest.skip("library not built by xla_amd.build in this tree")
  kernels = json.load(open(build.RESOURCES_PATH))
  assert len(kernels) > 50
  assert [k for k in kernels if k.get("scratch_bytes_per_lane", 0) > 0] == []


def test_headline_kernels_keep_their_code_budget():
  """The build records every kernel's code bytes; the decode kernels, whose cold prologue is part of every launch, have a budget."""
  import json
  from xla_amd import build
  if not os.path.exists(build.RESOURCES_PATH):
    pytest.skip("library not built by xla_amd.build in this tree")
  by_name = {k["kernel"]: k for k in json.load(open(build.RESOURCES_PATH))}
  assert all("code_bytes" in k and k["code_bytes"] > 0 for k in by_name.values())
  for name, budget in build.CODE_BUDGET_BYTES.items():
    assert name in by_name, name
    assert by_name[name]["code_bytes"] <= budget, (name, by_name[name]["code_bytes"], budget)


def test_a_replaced_library_replaces_the_operators_kernels():
  """A program that names another build of the library (the diagnostic one) gets that build's kernels from the operators
  too: the native operators, which are linked against the ordinary build, stay out of the process."""
  code = """
import os, torch
from xla_amd import _lib
_lib._LIB_PATH = os.path.join(os.path.dirname(_lib._LIB_PATH), "libxla_amd_qmm_timeline.so")
import xla_amd.experimental.xla_quantized_matmul as q
maps = open("/proc/self/maps").read()
_lib.load()
assert "libxla_amd_qmm_timeline.so" in open("/proc/self/maps").read()
assert "libxla_amd_qmm.so" not in maps and "libxla_amd_torch.so" not in maps
for op in ("xla::quantized_matmul", "xla_amd::weight_only_tiled"):
  assert torch._C._dispatch_has_kernel_for_dispatch_key(op, "CUDA")
assert q.counters.native is None and q.counters["pack"] == 0
"""
  subprocess.run([sys.executable, "-c", code], check=True, cwd=ROOT, timeout=120)
