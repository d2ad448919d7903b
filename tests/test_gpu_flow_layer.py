"""The fused sampling layer at batch sizes that leave a block's 64 rows part empty, for
every unrolled bin count and hidden width, in 8 and 14 dimensions.

A point does not depend on the points beside it, so a short pass has the bits of the first
points of a long one. The unrolled splines (two lanes each) do the operations of the
runtime loops (one lane) in the same order; what the compiler fuses may differ, one
rounding of 6e-8 an operation: 1e-6 in u, the bound of the two paths' other comparison,
and in x, which is u on a grid of equal bins."""
import ctypes as C

import numpy as np
import pytest

from graniitti_amd import abi
from graniitti_amd.process import MContinuum
from test_gpu_flow import flow_cfg, init_random

pytestmark = pytest.mark.gpu


def sample(P, n):
    w, x = np.empty(n), np.empty((n, P.cfg.dim))
    s = abi.GraFlowStats()
    abi.check(P.lib.gra_hip_flow_sample(P.h, n, 51, abi.dptr(w), abi.dptr(x), C.byref(s)), P.h)
    return w, x


@pytest.mark.parametrize("preset", [1, 3])
@pytest.mark.parametrize("H", [64, 128, 256])
@pytest.mark.parametrize("K", [8, 16, 32])
def test_ragged_batches(preset, H, K):
    cfg = abi.cfg_default(preset)
    cfg.screening = 0
    g = abi.GraGrid()
    abi.check(abi.load().gra_hip_grid_init(C.byref(g), cfg.dim, 128))
    print(f"case: fused layer D={cfg.dim} K={K} H={H}, 1, 63, 65, 257 points", flush=True)
    x = {}
    with MContinuum(cfg) as P:
        for loops in (1, 0):
            fc = flow_cfg(cfg.dim, 2, K, H, 2, False)
            fc.spline_loops = loops
            init_random(P, fc, 0.05, 41)
            abi.check(P.lib.gra_hip_flow_set_grid(P.h, C.byref(g)), P.h)
            w, x[loops] = sample(P, 257)
        for n in (1, 63, 65):
            wn, xn = sample(P, n)
            assert np.array_equal(wn, w[:n]) and np.array_equal(xn, x[0][:n]), n
    assert np.abs(x[0] - x[1]).max() <= 1e-6
