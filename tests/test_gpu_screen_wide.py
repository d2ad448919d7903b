"""Screening launches with few candidates, which take more lanes a candidate, against the
same points in a launch with many, for every node the screening kernels have.

Bounds. The FP32 Regge and tensor nodes keep the order of their rounded sums: the same
bits. The other nodes are summed in FP64 in another order: 500 roundings of 1e-16, in a
screened amplitude that can be 1/10 of its parts, squared: 1e-12."""
import numpy as np
import pytest

from graniitti_amd import abi
from graniitti_amd.process import MContinuum
from conftest import small_tables

pytestmark = pytest.mark.gpu

F32, F64 = abi.GRA_AMP_FP32, abi.GRA_AMP_FP64
NODES = {
    # name: (preset, amplitude, overrides, points of the large launch, bound)
    "regge_fp32": (2, F32, {}, 60000, 0.0),
    "regge_fp64": (2, F64, {"offshellFF": 0}, 20000, 1e-12),
    "regge_folded": (2, F64, {}, 20000, 1e-12),
    "resonances": (7, F64, {"spin_frame": abi.GRA_FRAME_GJ}, 20000, 1e-12),
    "resonances_folded": (7, F64, {}, 20000, 1e-12),
    "resonances_folded_fp32": (7, F32, {}, 20000, 1e-12),
    "tensor_2xs": (10, F64, {}, 20000, 1e-12),
    "tensor_fp64": (3, F64, {}, 20000, 1e-12),
    "tensor_fp32": (3, F32, {}, 20000, 0.0),
}


@pytest.mark.parametrize("loop", [(15, 30), (21, 9)])
@pytest.mark.parametrize("name", sorted(NODES))
def test_few_candidates(name, loop):
    preset, amp, over, n, bound = NODES[name]
    cfg = small_tables(abi.cfg_default(preset), 500)
    cfg.screening, cfg.amp_precision = 1, amp
    cfg.n_loop_phi, cfg.n_loop_kt = loop
    for key, value in over.items():
        setattr(cfg, key, value)
    print(f"case: {name}, loop {loop}, 1, 5, 67 points against {n}", flush=True)
    u = np.random.default_rng(91).random((n, cfg.dim))
    with MContinuum(cfg) as P:
        W, a, f = P.eval(u)
        for k in (1, 5, 67):
            Wk, ak, fk = P.eval(u[:k])
            assert np.array_equal(fk, f[:k]), k
            np.testing.assert_allclose(Wk, W[:k], rtol=bound, atol=0, err_msg=str(k))
            np.testing.assert_allclose(ak, a[:k], rtol=bound, atol=0, err_msg=str(k))
    assert np.count_nonzero(W[:67]) > 10
