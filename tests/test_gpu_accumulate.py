"""One VEGAS iteration's sums and histograms against the oracle at the sizes where the
accumulation's splits leave remainders: batches of 64 points, blocks of 512, runs of
lanes that share a bin (two bins in a dimension: every lane has about 32 others), 8 and
14 dimensions on waves that own dimensions in turn.

Tolerance. A weight agrees with the oracle's to 1e-10 (continuum) or 1e-9 (tensor pair),
the bounds of the pointwise tests; every term of a sum is positive, so a sum of f agrees
as its terms do, a sum of f^2 to twice that; the rounding of up to 5000 additions, 1e-12,
is far below."""
import ctypes as C

import numpy as np
import pytest

from graniitti_amd import abi
from graniitti_amd.process import MContinuum
import oracle_lib as ol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("preset,rtol", [(1, 1e-10), (3, 1e-9)])
@pytest.mark.parametrize("bins", [2, 16, 128])
@pytest.mark.parametrize("n", [1, 63, 65, 511, 513, 4097])
def test_iteration_sums(preset, rtol, bins, n):
    cfg = abi.cfg_default(preset)
    cfg.screening, cfg.amp_precision = 0, abi.GRA_AMP_FP64
    g = abi.GraGrid()
    abi.check(abi.load().gra_hip_grid_init(C.byref(g), cfg.dim, bins))
    print(f"case: preset {preset}, {cfg.dim} dimensions, {bins} bins, {n} points", flush=True)
    with MContinuum(cfg) as P:
        sg = P.vegas_iterate(g, n, 41, 2)
    so = ol.OracleRun(cfg).vegas_iterate(g, n, 41, 2)
    for k in ("n_calls", "n_kin_ok", "n_fid_ok", "n_valid", "n_nan", "n_inf"):
        assert getattr(sg, k) == getattr(so, k), k
    for k in ("fsum", "maxW", "maxf"):
        assert abs(getattr(sg, k) - getattr(so, k)) <= rtol * getattr(so, k), k
    assert abs(sg.f2sum - so.f2sum) <= 2 * rtol * so.f2sum
    for k, tol in (("fmat", rtol), ("f2mat", 2 * rtol)):
        np.testing.assert_allclose(np.ctypeslib.as_array(getattr(sg, k)),
                                   np.ctypeslib.as_array(getattr(so, k)), rtol=tol, atol=0,
                                   err_msg=k)
