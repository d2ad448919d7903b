"""One VEGAS iteration's sums and histograms against the oracle where the reduction of the
block partials leaves its short forms: 512 partials (16 loads in flight for each of the 32
groups, one turn of the scalars' threads), one more (remainders and a second turn), and the
8192 partials beyond which blocks grow instead.

Tolerances as in test_gpu_accumulate.py, with 4e6 additions of positive terms: 1e-10 of each
term, the rounding of the sums (blocks of 512 terms, 8192 blocks in 32 groups) 1e-13."""
import ctypes as C

import numpy as np
import pytest

from graniitti_amd import abi
from graniitti_amd.process import MContinuum
import oracle_lib as ol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("preset,n,rtol", [(1, 512 * 512, 1e-10), (1, 512 * 512 + 1, 1e-10),
                                           (1, 512 * 1055 + 77, 1e-10), (3, 512 * 530 + 3, 1e-9),
                                           (1, 512 * 8192 + 777, 1e-10)])
def test_iteration_sums(preset, n, rtol):
    cfg = abi.cfg_default(preset)
    cfg.screening, cfg.amp_precision = 0, abi.GRA_AMP_FP64
    g = abi.GraGrid()
    abi.check(abi.load().gra_hip_grid_init(C.byref(g), cfg.dim, 128))
    print(f"case: preset {preset}, {cfg.dim} dimensions, {n} points", flush=True)
    with MContinuum(cfg) as P:
        sg = P.vegas_iterate(g, n, 43, 1)
    print("iteration done", flush=True)
    so = ol.OracleRun(cfg).vegas_iterate(g, n, 43, 1)
    for k in ("n_calls", "n_kin_ok", "n_fid_ok", "n_valid", "n_nan", "n_inf"):
        assert getattr(sg, k) == getattr(so, k), k
    for k in ("fsum", "maxW", "maxf"):
        assert abs(getattr(sg, k) - getattr(so, k)) <= rtol * getattr(so, k), k
    assert abs(sg.f2sum - so.f2sum) <= 2 * rtol * so.f2sum
    for k, tol in (("fmat", rtol), ("f2mat", 2 * rtol)):
        np.testing.assert_allclose(np.ctypeslib.as_array(getattr(sg, k)),
                                   np.ctypeslib.as_array(getattr(so, k)), rtol=tol, atol=0,
                                   err_msg=k)
