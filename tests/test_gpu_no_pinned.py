"""Small evaluations and VEGAS iterations where no pinned memory is to be had for the
handle's buffer: the same results, bit for bit, through device buffers.

A child process loads, before the library, a definition of hipHostMalloc that refuses the
sizes of that buffer (64 kB and more) and passes smaller ones on to the runtime's."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static long refused;
extern "C" long refusals() { return refused; }
extern "C" int hipHostMalloc(void** p, size_t n, unsigned flags) {
  typedef int (*fn)(void**, size_t, unsigned);
  static fn real = (fn)dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY), "hipHostMalloc");
  if (n < 65536) return real(p, n, flags);
  ++refused;
  *p = nullptr;
  return 2;  // hipErrorOutOfMemory
}
"""

CHILD = r"""
import ctypes as C, sys
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
shim = C.CDLL(sys.argv[3], mode=C.RTLD_GLOBAL) if len(sys.argv) > 3 else None
import numpy as np
from graniitti_amd import abi
from graniitti_amd.process import MContinuum
out = {}
for preset in (1, 3):
    cfg = abi.cfg_default(preset)
    cfg.screening = 0
    g = abi.GraGrid()
    abi.check(abi.load().gra_hip_grid_init(C.byref(g), cfg.dim, 64))
    u = np.random.default_rng(6).random((777, cfg.dim))
    print("case: preset", preset, flush=True)
    with MContinuum(cfg) as P:
        for k in range(2):
            out[f"W{preset}{k}"], out[f"a{preset}{k}"], out[f"f{preset}{k}"] = P.eval(u)
            st = P.vegas_iterate(g, 3001, 5, k)
            out[f"s{preset}{k}"] = np.frombuffer(bytes(st), np.uint8)
if shim is not None:
    shim.refusals.restype = C.c_long
    assert shim.refusals() >= 4, "the buffer was not refused"
np.savez(sys.argv[2], **out)
"""


def test_without_pinned_memory(tmp_path):
    src, shim = tmp_path / "shim.cpp", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", str(src), "-o", str(shim), "-ldl"], check=True)
    got = []
    for extra in ([], [str(shim)]):
        npz = str(tmp_path / f"r{len(extra)}.npz")
        p = subprocess.run([sys.executable, "-c", CHILD, ROOT, npz] + extra, cwd=ROOT, text=True,
                           capture_output=True, timeout=100)
        print(p.stdout, p.stderr, flush=True)
        assert p.returncode == 0
        got.append(np.load(npz))
    assert len(got[0].files) == 16
    for k in got[0].files:
        np.testing.assert_array_equal(got[0][k], got[1][k], err_msg=k)
