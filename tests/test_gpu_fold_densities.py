"""Point-folded resonance nodes with several spin densities a spin: every class of density
and trace that a point can have, the largest number of sums, and densities that return
after another one. test_gpu_fold.py has one density a spin there, or off-diagonal ones,
which keep the reference-order nodes.

That a case is folded is shown by the same run with one off-diagonal pair of 1e-300 a
density: it changes no bit of a reference-order node, but sends the run to those nodes.

Tolerances: those of test_gpu_fold.py, against the oracle (FP64) or the general FP64 nodes
(FP32 amplitude), and between the two forms of node."""
import numpy as np
import pytest

from graniitti_amd import abi
from graniitti_amd.process import MContinuum
from conftest import small_tables
import oracle_lib as ol

pytestmark = pytest.mark.gpu

F32, F64 = abi.GRA_AMP_FP32, abi.GRA_AMP_FP64
TOL = {F64: 2e-10, F32: 6e-5}
# diagonals, by spin; unequal at +-m, and with and without the row m = 0
D1 = [(0.5, 0.0, 0.5), (0.2, 0.5, 0.3), (0.0, 1.0, 0.0), (0.6, 0.1, 0.3)]
D2 = [(0.5, 0.0, 0.0, 0.0, 0.5), (0.1, 0.2, 0.4, 0.2, 0.1), (0.3, 0.0, 0.5, 0.1, 0.1),
      (0.0, 0.5, 0.0, 0.5, 0.0), (0.0, 0.0, 1.0, 0.0, 0.0), (0.2, 0.2, 0.2, 0.2, 0.2),
      (0.25, 0.25, 0.1, 0.15, 0.25), (0.4, 0.1, 0.0, 0.1, 0.4)]
# name: the spin and density of each resonance
SETS = {
    "tensors_8": [(2, k) for k in range(8)],
    "vectors_2": [(1, 0), (1, 1)],
    "vectors_return": [(1, 1), (1, 2), (1, 1), (1, 3)],
    "tensors_return": [(2, 1), (2, 2), (2, 1), (2, 5)],
    "mixed": [(2, 1), (1, 3), (0, 0), (2, 3), (1, 1), (2, 1), (1, 3), (0, 0)],
    "mixed_8": [(1, 0), (1, 1), (1, 2), (1, 3), (2, 4), (2, 5), (2, 6), (2, 7)],
}


def config(name, amp):
    cfg = small_tables(abi.cfg_default(7), 500)
    cfg.amp_precision = amp
    src = {J: [abi.GraRes.from_buffer_copy(cfg.res[r]) for r in range(cfg.n_res)
               if cfg.res[r].J == J] for J in (0, 1, 2)}
    for r, (J, d) in enumerate(SETS[name]):
        q = abi.GraRes.from_buffer_copy(src[J][r % len(src[J])])
        q.mass += 0.05 * r  # no two alike
        if J:
            diag, n = (D1 if J == 1 else D2)[d], 2 * J + 1
            for k in range(n * n):
                q.rho_re[k] = diag[k // n] if k % (n + 1) == 0 else 0.0
                q.rho_im[k] = 0.0
        cfg.res[r] = q
    cfg.n_res = len(SETS[name])
    return cfg


def off_diagonal(cfg):
    c = abi.GraCfg.from_buffer_copy(cfg)
    for r in range(c.n_res):
        if c.res[r].J:
            c.res[r].rho_re[1] = c.res[r].rho_re[2 * c.res[r].J + 1] = 1e-300
    return c


def weights(cfg, u):
    with MContinuum(cfg) as P:
        return P.eval(u)


@pytest.mark.parametrize("over", [{}, {"spin_frame": abi.GRA_FRAME_HX, "spin_dec": 0},
                                  {"spin_gen": 0}, {"process": abi.GRA_PROC_RES}],
                         ids=["collins_soper", "helicity_no_decay", "no_production", "no_continuum"])
@pytest.mark.parametrize("amp", [F64, F32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("name", sorted(SETS))
def test_densities(name, amp, over):
    cfg = config(name, amp)
    for key, value in over.items():
        setattr(cfg, key, value)
    general = off_diagonal(cfg)
    n = 65 if amp == F64 else 513
    print(f"case: {name}, {over}, amplitude {amp}, {n} points", flush=True)
    u = np.random.default_rng(73).random((n, cfg.dim))
    W, _, f = weights(cfg, u)
    Wn, _, fn = weights(general, u)
    # the FP32 amplitude's reference: the general FP64 nodes, held to the oracle above
    ref = abi.GraCfg.from_buffer_copy(cfg if amp == F64 else general)
    ref.amp_precision = F64
    Wo, _, fo = ol.OracleRun(ref).eval(u) if amp == F64 else weights(ref, u)
    assert np.array_equal(f, fo) and np.array_equal(fn, fo)
    assert not np.array_equal(W, Wn), "not folded"
    # FP32 resolves the weights above 1e-8 of the largest
    big = Wo > (1e-8 * Wo.max() if amp == F32 else 0.0)
    assert big.sum() > 10
    for a, b, what in ((W, Wo, "folded, reference"), (W, Wn, "folded, general")):
        rel = np.abs(a[big] - b[big]) / Wo[big]
        print(f"{what}: max rel {rel.max():.2e}", flush=True)
        assert rel.max() <= TOL[amp], what


@pytest.mark.parametrize("amp", [F64, F32], ids=["fp64", "fp32"])
def test_the_off_diagonal_pair_changes_no_bit(amp):
    """In the Gottfried-Jackson frame, where both runs take reference-order nodes."""
    cfg = config("mixed", amp)
    cfg.spin_frame = abi.GRA_FRAME_GJ
    print(f"case: Gottfried-Jackson, amplitude {amp}, 65 points", flush=True)
    u = np.random.default_rng(74).random((65, cfg.dim))
    assert np.array_equal(weights(cfg, u)[0], weights(off_diagonal(cfg), u)[0])
