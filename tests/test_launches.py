"""What the library's entry points launch, recorded without a GPU."""
import pytest

from tests import launch_recorder as rec


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
