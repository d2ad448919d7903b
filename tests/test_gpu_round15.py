"""The eikonal tables' rows as the table kernel rounds them: every value is the one that
writing it with 15 digits and reading it back gives. Exact."""
import numpy as np
import pytest

from graniitti_amd import abi
from graniitti_amd.process import MContinuum
from conftest import small_tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("beam,rows", [(6500.0, 500), (6500.0, 10000), (100.0, 501), (31.0, 63)])
def test_rows_are_rounded(beam, rows):
    cfg = small_tables(abi.cfg_default(2), rows)
    cfg.n_fb = rows + rows % 2  # Simpson's rule takes an even number
    cfg.beam_E1 = cfg.beam_E2 = beam
    print(f"case: tables of {rows} intervals, beams of {beam} GeV", flush=True)
    with MContinuum(cfg) as P:
        _, mbt, msa = P.eikonal_tables()
    for T in (mbt, msa):
        text = np.array([float("%.15g" % v) for v in T.ravel()]).reshape(T.shape)
        assert np.array_equal(T, text)
