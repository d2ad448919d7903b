"""A point's weight does not depend on its call: the screening kernels take more lanes a
candidate in a launch with few candidates (up to 8192 in the FP64 unit and 32768 for the FP32
Regge node; 16384 points for the FP32 tensor node), on both sides of which every node they
have gives the same bits."""
import numpy as np
import pytest

from graniitti_amd import abi
from graniitti_amd.process import MContinuum
from conftest import small_tables

pytestmark = pytest.mark.gpu

F32, F64 = abi.GRA_AMP_FP32, abi.GRA_AMP_FP64
NODES = {
    # name: (preset, amplitude, overrides, points of the large launch)
    "regge_fp32": (2, F32, {}, 50001),
    "regge_fp64": (2, F64, {"offshellFF": 0}, 20001),
    "regge_folded": (2, F64, {}, 20001),
    "factorized_folded": (5, F64, {}, 30001),
    "gauss_folded": (11, F64, {}, 20001),
    "resonances": (7, F64, {"spin_frame": abi.GRA_FRAME_GJ}, 20001),
    "resonances_fp32": (7, F32, {"spin_frame": abi.GRA_FRAME_GJ}, 20001),
    "resonances_folded": (7, F64, {}, 20001),
    "resonances_folded_fp32": (7, F32, {}, 20001),
    "tensor_2xs": (10, F64, {}, 20001),
    "tensor_fp64": (3, F64, {}, 20001),
    "tensor_fp32": (3, F32, {}, 20001),
}


@pytest.mark.parametrize("loop", [(15, 30), (21, 9)])
@pytest.mark.parametrize("name", sorted(NODES))
def test_weight_does_not_depend_on_call(name, loop):
    preset, amp, over, n = NODES[name]
    cfg = small_tables(abi.cfg_default(preset), 500)
    cfg.screening, cfg.amp_precision = 1, amp
    cfg.n_loop_phi, cfg.n_loop_kt = loop
    for key, value in over.items():
        setattr(cfg, key, value)
    print(f"case: {name}, loop {loop}, 1, 5, 67, 4999 points against {n}", flush=True)
    u = np.random.default_rng(92).random((n, cfg.dim))
    with MContinuum(cfg) as P:
        W, a, f = P.eval(u)
        for k in (1, 5, 67, 4999):
            Wk, ak, fk = P.eval(u[:k])
            for got, all_ in ((Wk, W), (ak, a), (fk, f)):
                np.testing.assert_array_equal(got, all_[:k], err_msg=str(k))
    assert np.count_nonzero(W[:67]) > 5
