"""Evaluation of host points on both sides of the size up to which the kernels read and
write the handle's pinned buffer (81 bytes a point in 8 dimensions of 512 kB: 6472 points,
beyond it device copies), and from one size to another on one handle.

A point's weight does not depend on its call: all comparisons are of bits."""
import numpy as np
import pytest

from graniitti_amd import abi
from graniitti_amd.process import MContinuum
from conftest import small_tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("preset", [1, 2])
def test_sizes_on_one_handle(preset):
    cfg = small_tables(abi.cfg_default(preset), 500)
    print(f"case: preset {preset}, 1 to 9001 points, up and down on one handle", flush=True)
    u = np.random.default_rng(81).random((9001, cfg.dim))
    with MContinuum(cfg) as P:
        W, a, f = P.eval(u)
        for n in (1, 1000, 6472, 6473, 9001, 2, 6472):
            Wn, an, fn = P.eval(u[:n])
            assert np.array_equal(Wn, W[:n]) and np.array_equal(an, a[:n]), n
            assert np.array_equal(fn, f[:n]), n
        # results that the caller does not want
        Wn = np.empty(500)
        abi.check(P.lib.gra_hip_eval_points(P.h, abi.dptr(np.ascontiguousarray(u[:500])), 500,
                                            abi.dptr(Wn), None, None), P.h)
        assert np.array_equal(Wn, W[:500])
