"""Which kernels a call of the library launches, and how, without a GPU: tests/launch_recorder.cpp takes the place of
the HIP runtime in a process of its own.  Pointers handed to the calls are never read."""
import collections
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

# name: the kernel's (mangled) device name; lds, lds_limit: dynamic LDS asked for, and allowed for that kernel; args: the
# first words of the kernel's argument struct
Launch = collections.namedtuple("Launch", "name grid block lds lds_limit args")

_CHILD = """
import ctypes, json, sys
rec = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # in front of the runtime in every later lookup
lib = ctypes.CDLL(sys.argv[2])
rec.take_notes.restype = lib.xla_amd_qmm_last_error.restype = ctypes.c_char_p
types = {"p": ctypes.c_void_p, "q": ctypes.c_int64, "i": ctypes.c_int, "z": ctypes.c_size_t}
out = []
for name, sig, args in json.load(sys.stdin):
  fn = getattr(lib, name)
  fn.argtypes = [types[c] for c in sig]
  rc = fn(*args)
  out.append((rc, lib.xla_amd_qmm_last_error().decode() if rc else "", rec.take_notes().decode()))
json.dump(out, sys.stdout)
"""


def record(calls, workdir):
  """calls: (function, one letter per argument - p pointer, q int64, i int, z size -, arguments), made in order in one
  process.  Returns (return code, error text, launches) for each."""
  shim = os.path.join(workdir, "recorder.so")
  subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-shared", "-fPIC",
                  os.path.join(HERE, "launch_recorder.cpp"), "-o", shim], check=True)
  lib = os.path.join(ROOT, "xla_amd", "libxla_amd_qmm.so")
  got = subprocess.run([sys.executable, "-c", _CHILD, shim, lib], input=json.dumps(calls), capture_output=True, text=True,
                       timeout=120)
  assert got.returncode == 0, got.stderr
  out = []
  for rc, text, notes in json.loads(got.stdout):
    launches = []
    for line in notes.splitlines():
      name, *n = line.split()
      n = [int(v) for v in n]
      launches.append(Launch(name, tuple(n[0:3]), tuple(n[3:6]), n[6], n[7], n[8:]))
    out.append((rc, text, launches))
  return out


PTR = 1 << 20  # an aligned address for arguments that are not looked at


def generic(m, n, k, zp=False, x_dt=1):
  dts = [x_dt] * 6
  return ("xla_amd_qmm_weight_only_generic", "ppppp" + "qqqq" + "iiiiiii" + "p",
          [PTR, PTR, PTR, PTR if zp else 0, PTR, m, n, k, k, 0, *dts, 0])


def w8a8(m, n, k, block_m=0, block_n=0, out_dt=1):
  return ("xla_amd_qmm_w8a8_gemm", "p" * 8 + "qqq" + "i" * 9 + "p",
          [PTR, PTR, PTR, PTR, 0, 0, PTR, 0, m, n, k, 0, 0, 0, 0, 0, 0, out_dt, block_m, block_n, 0])


def blockwise(m, n, k, c, bits, zp, x_dt=1):
  return ("xla_amd_qmm_weight_only_gemm", "pppppp" + "z" + "qqqq" + "iiiiiii" + "p",
          [PTR, PTR, PTR, PTR if zp else 0, PTR, PTR, 1 << 40, m, n, k, c, bits, *[x_dt] * 6, 0])


def skinny(m, n, k, c, bits, zp, x_dt=1):
  return ("xla_amd_qmm_weight_only_skinny", "ppppp" + "qqqq" + "iiiiiii" + "p",
          [PTR, PTR, PTR, PTR if zp else 0, PTR, m, n, k, c, bits, *[x_dt] * 6, 0])


def gemm_f32(m, n, k, zp=False, workspace=PTR, workspace_bytes=1 << 40):
  return ("xla_amd_qmm_weight_only_gemm_f32", "pppppp" + "z" + "qqq" + "iip",
          [PTR, PTR, PTR, PTR if zp else 0, PTR, workspace, workspace_bytes, m, n, k, 0, 0, 0])
