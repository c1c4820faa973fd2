"""The native operator implementations against the Python formulation of the same operators."""
import gc
import threading

import pytest
import torch

from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
  import xla_amd.experimental.xla_quantized_matmul as q
  assert q.counters.native is not None, "libxla_amd_torch.so is not built"
  return q


native = lambda *a: torch.ops.xla.quantized_matmul(*a)
general = lambda *a: torch.ops.xla_amd.quantized_matmul_general(*a)


def _outcome(fn, args):
  try:
    return fn(*args)
  except Exception as e:  # noqa: BLE001  (the same refusal is the point)
    return type(e), str(e).split("\n")[0]


def _same(args):
  a, b = _outcome(native, args), _outcome(general, args)
  if isinstance(b, tuple):
    assert a == b
  else:
    assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)


def test_same_calls_same_answers(ops):
  k, n = 256, 192
  for xdt in (torch.float32, torch.bfloat16, torch.float16):
    for sdt in (torch.float32, xdt):
      for m in (1, 17, 40, 130):
        x, w, s, _ = cases.per_channel_int8(m, n, k, xdt, sdt, seed=m)
        x, w, s = x.cuda(), w.cuda(), s.cuda()
        z = (torch.randn(n, device="cuda") * 0.01).to(sdt)
        for zp in (None, z):
          for act in (False, True):
            _same((x, w, s, zp, -1, False, act))
        _same((x, w.clamp(-8, 7), s, z, -1, True, False))
        # layouts: rows of a wider tensor, columns first, three and one dimensions, none, strided weight and scale
        wide = torch.zeros(m, k + 8, dtype=xdt, device="cuda")
        wide[:, :k] = x
        for xs in (wide[:, :k], x.t().contiguous().t(), x.reshape(1, m, k), x[0], x[:0]):
          _same((xs, w, s, z, -1, False, False))
          if xs.dim() == 2:
            _same((xs, w, s, z, -1, False, True))
        wt = w.t().contiguous().t()
        _same((x, wt, s, None, -1, False, False))
        _same((x, wt, s, None, -1, False, True))
        s2 = torch.stack([s, s], 1)[:, 0]
        _same((x, w, s2, s2, -1, False, False))
      x, w, s, z, _ = cases.blockwise(33, n, k, 128, 4, xdt, seed=1)
      for sc, zp in ((s, z), (s, None), (s.to(sdt), z.to(sdt))):  # (mixed dtypes are refused)
        for bits4 in (True, False):
          _same((x.cuda(), w.cuda(), sc.cuda(), zp if zp is None else zp.cuda(), 128, bits4, False))
      # odd K: the operator's own layouts, one block of all of K among them
      x, w, s, z, _ = cases.blockwise(9, 52, 77, 77, 8, xdt, seed=3)
      _same((x.cuda(), w.cuda(), s.cuda(), z.cuda(), 77, False, False))
      x, w, s, z, _ = cases.blockwise(9, 52, 90, 30, 8, xdt, seed=3)
      _same((x.cuda(), w.cuda(), s.cuda(), z.cuda(), 30, False, False))
      x, w, s, _ = cases.per_channel_int8(9, 50, 77, xdt, sdt, seed=2)
      _same((x.cuda(), w.cuda(), s.cuda(), None, -1, False, False))


def test_same_refusals(ops):
  x, w, s, _ = cases.per_channel_int8(4, 64, 128, torch.bfloat16, torch.bfloat16)
  x, w, s = x.cuda(), w.cuda(), s.cuda()
  for args in ((x, w.float(), s, None, -1, False, False), (x, w[:, :64], s, None, -1, False, False),
               (x, w, s[:32], None, -1, False, False), (x, w, s, None, 128, False, False),
               (x, w, s, None, 128, False, True), (x, w[None], s, None, -1, False, False), (x.double(), w, s, None, -1, False, False),
               (x, w, s.double(), None, -1, False, False), (x.int(), w, s, None, -1, False, False), (x, w, s, None, 0, False, False),
               (x, w.t().reshape(2, 64, 64), torch.stack([s, s]).float(), None, 64, False, False)):
    _same(args)
    assert isinstance(_outcome(native, args), tuple)


def test_overflow_policy(ops, monkeypatch):
  x, w, s, _ = cases.per_channel_int8(40, 64, 128, torch.bfloat16, torch.bfloat16)
  for policy in ("wrap", "saturate", "neither"):
    monkeypatch.setenv("XLA_AMD_QMM_OVERFLOW", policy)
    _same((x.cuda(), w.cuda(), s.cuda(), None, -1, False, True))


def test_copies_follow_their_weights(ops):
  x, w, s, _ = cases.per_channel_int8(4, 4096, 4096, torch.bfloat16, torch.bfloat16)
  x, w, s = x.cuda(), w.cuda(), s.cuda()
  args = lambda: (x, w, s, None, -1, False, False)
  native(*args())
  before = dict(ops.counters)
  native(*args())
  assert ops.counters["pack_hit"] == before["pack_hit"] + 1 and ops.counters["pack"] == before["pack"]
  w.neg_()  # seen through the version counter
  first = native(*args())
  assert ops.counters["pack"] == before["pack"] + 1
  assert torch.equal(first, general(x, w.clone(), s, None, -1, False, False))
  w.data.neg_()  # not seen: the call below says so
  ops.invalidate_weight_cache(w)
  assert torch.equal(native(*args()), general(x, w.clone(), s, None, -1, False, False))
  # int4 and int8 readings of one container do not share a copy
  w.clamp_(-8, 7)
  a, b = native(x, w, s, None, -1, True, False), native(x, w, s, None, -1, False, False)
  assert cases.rel_l2(a.cpu(), b.cpu()) < 1e-2
  # the copy goes with its weight
  gc.collect()
  held = torch.cuda.memory_allocated()
  del w
  gc.collect()
  assert held - torch.cuda.memory_allocated() >= 2 * 4096 * 4096


def test_threads_and_streams(ops):
  """Several threads, each on a stream of its own, with weights of their own and a shared one."""
  x, w, s, _ = cases.per_channel_int8(33, 512, 1024, torch.bfloat16, torch.bfloat16)
  x, s, shared = x.cuda(), s.cuda(), w.cuda()
  want = general(x, shared, s, None, -1, False, False)
  torch.cuda.synchronize()
  wrong = []

  def work():
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
      for _ in range(20):
        own = shared.clone()
        for got in (native(x, own, s, None, -1, False, False), native(x, shared, s, None, -1, False, False)):
          if not torch.equal(got, want):
            wrong.append(1)
    st.synchronize()

  threads = [threading.Thread(target=work) for _ in range(4)]
  for t in threads:
    t.start()
  for t in threads:
    t.join()
  assert not wrong


def _busy(stream, ms=60):
  with torch.cuda.stream(stream):
    torch.cuda._sleep(int(ms * 2.4e6))  # (cycles)


@pytest.mark.parametrize("call", [native, general])
def test_copy_made_on_another_stream(ops, call):
  """A weight's first call on one stream, its second on another: the second waits for the copy the first is making."""
  x, w, s, _ = cases.per_channel_int8(33, 512, 1024, torch.bfloat16, torch.bfloat16)
  x, s, w = x.cuda(), s.cuda(), w.cuda()
  want = call(x, w.clone(), s, None, -1, False, False)
  first, second = torch.cuda.Stream(), torch.cuda.Stream()
  torch.cuda.synchronize()
  _busy(first)
  with torch.cuda.stream(first):
    a = call(x, w, s, None, -1, False, False)
  with torch.cuda.stream(second):
    b = call(x, w, s, None, -1, False, False)
  assert not first.query()  # (both calls were made while the copy was still to come)
  second.synchronize()
  assert torch.equal(b, want)
  torch.cuda.synchronize()
  assert torch.equal(a, want)


@pytest.mark.parametrize("call", [native, general])
def test_copy_replaced_under_another_stream(ops, call):
  """A copy that is replaced (an in-place write to its weight) while another stream still has to read it keeps its
  memory until then."""
  x, w, s, _ = cases.per_channel_int8(33, 512, 1024, torch.bfloat16, torch.bfloat16)
  x, s, w = x.cuda(), s.cuda(), w.cuda()
  want = call(x, w, s, None, -1, False, False)
  size = ops._pack_cache[(id(w), "tiled")][3].numel()
  other = torch.cuda.Stream()
  with torch.cuda.stream(other):
    call(x, w, s, None, -1, False, False)
  # (memory the calls below take without going to the driver, which may wait for the whole device)
  del [torch.empty(size, dtype=torch.uint8, device="cuda") for _ in range(16)][:]
  torch.cuda.synchronize()
  _busy(other)
  with torch.cuda.stream(other):
    a = call(x, w, s, None, -1, False, False)
  w.neg_()
  call(x, w, s, None, -1, False, False)  # makes the new copy, lets go of the old one
  taken = [torch.full((size,), 99, dtype=torch.uint8, device="cuda") for _ in range(8)]
  assert not other.query()  # (all of this was launched before the read; where the streams share a hardware queue it also runs in that order)
  torch.cuda.synchronize()
  assert torch.equal(a, want)
  del taken


@pytest.mark.parametrize("call", [native, general])
def test_copy_still_being_made_at_a_capture(ops, call):
  """A capture on another stream than the one that is making the copy: the graph finds it complete."""
  x, w, s, _ = cases.per_channel_int8(33, 512, 1024, torch.bfloat16, torch.bfloat16)
  x, s, w = x.cuda(), s.cuda(), w.cuda()
  want = call(x, w.clone(), s, None, -1, False, False)
  first, second = torch.cuda.Stream(), torch.cuda.Stream()
  torch.cuda.synchronize()
  _busy(first)
  with torch.cuda.stream(first):
    call(x, w, s, None, -1, False, False)
  g = torch.cuda.CUDAGraph()
  with torch.cuda.stream(second):
    g.capture_begin()
    out = call(x, w, s, None, -1, False, False)
    g.capture_end()
    for _ in range(3):
      out.zero_()
      g.replay()
      second.synchronize()
      assert torch.equal(out, want)
