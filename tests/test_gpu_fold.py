"""The point-folded FP64 screening nodes (gra_fold.h, gra_fold_res.h) against the oracle's
reference-order loop, over what the dispatch sends there: both phase-space classes,
every off-shell form factor, both loop rules down to a single node, launches that do
not fill a wave or a block, the resonances' frames, spin switches and densities, and
runs outside the form's range (low beams, few nodes, other form factors, the
Gottfried-Jackson frame), which keep the reference-order nodes.

Tolerance. Folded and reference-order nodes differ by the rounding of the component
form: t1, t2, t^ and u^ carry about 1e-12 GeV^2 of noise from node to node (E eps
times an energy transfer of a few GeV), which the amplitude sees with slopes below 10
per GeV^2, and a screened amplitude can be 1/10 of its tree and loop parts, squared:
1e-12 x 10 x 10 x 2 = 2e-10."""
import sys

import numpy as np
import pytest

from graniitti_amd import abi
from graniitti_amd.process import MContinuum
from conftest import small_tables
import oracle_lib as ol

pytestmark = pytest.mark.gpu

RTOL = 2e-10

CASES = {
    # name: (preset, points, overrides)
    "one_point": (2, 3, {}),
    "continuum": (2, 257, {}),
    "exp_form_factor": (2, 65, {"offshellFF": 0}),
    "orear_form_factor": (2, 65, {"offshellFF": 1}),
    "other_scale_s0": (2, 65, {"regge_s0": 1.7}),
    "factorized": (5, 129, {}),
    "simpson_3x3": (2, 65, {"n_loop_phi": 3, "n_loop_kt": 3}),
    "simpson_30x30": (2, 33, {"n_loop_phi": 30, "n_loop_kt": 30}),
    "gauss_one_node": (11, 65, {"n_loop_phi": 0, "n_loop_kt": 0}),
    "gauss_2x5": (11, 65, {"n_loop_phi": 1, "n_loop_kt": 4}),
    "beams_3500": (2, 65, {"beam_E1": 3500.0, "beam_E2": 3500.0}),
    "beams_100": (2, 65, {"beam_E1": 100.0, "beam_E2": 100.0}),
}


def mixed_density(cfg):
    """Full complex spin densities, a different one for each resonance with J > 0."""
    rng = np.random.default_rng(5)
    for r in range(cfg.n_res):
        q = cfg.res[r]
        m = 2 * q.J + 1
        a = rng.normal(size=(m, m)) + 1j * rng.normal(size=(m, m))
        rho = a @ a.conj().T
        rho /= np.trace(rho).real
        for k, v in enumerate(rho.reshape(-1)):
            q.rho_re[k], q.rho_im[k] = v.real, v.imag


def one_photoproduced(cfg):
    """The rho(770) alone, beside the continuum."""
    cfg.res[0] = cfg.res[7]
    cfg.n_res = 1


def all_tensors(cfg):
    """Eight J = 2 resonances, each with its own density: the most sums a point can have."""
    for r in range(8):
        mass, width = cfg.res[r].mass, cfg.res[r].width
        cfg.res[r] = cfg.res[4]
        cfg.res[r].mass, cfg.res[r].width = mass, width
    mixed_density(cfg)


RES_CASES = {
    "res_collins_soper": ({}, None),
    "res_helicity": ({"spin_frame": abi.GRA_FRAME_HX}, None),
    "res_cm": ({"spin_frame": abi.GRA_FRAME_CM}, None),
    "res_no_production_spin": ({"spin_gen": 0}, None),
    "res_no_decay_spin": ({"spin_dec": 0}, None),
    "res_full_densities": ({}, mixed_density),
    "res_one_photoproduced": ({}, one_photoproduced),
    "res_all_tensors": ({}, all_tensors),
    "res_no_continuum": ({"process": abi.GRA_PROC_RES}, None),
    "res_none": ({"n_res": 0}, None),
}


@pytest.mark.parametrize("name", sorted(CASES) + sorted(RES_CASES))
def test_folded_nodes(name):
    change = None
    if name in CASES:
        preset, n, over = CASES[name]
    else:
        preset, n, (over, change) = 7, 65, RES_CASES[name]
    cfg = small_tables(abi.cfg_default(preset), 500)
    cfg.amp_precision = abi.GRA_AMP_FP64
    for key, value in over.items():
        setattr(cfg, key, value)
    if change:
        change(cfg)
    print(f"case: {name}, {n} points", flush=True)
    u = np.random.default_rng(71).random((n, cfg.dim))
    with MContinuum(cfg) as P:
        Wg, _, fg = P.eval(u)
    Wo, _, fo = ol.OracleRun(cfg).eval(u)
    ok = Wo != 0
    rel = np.abs(Wg[ok] - Wo[ok]) / Wo[ok]
    print(f"{ok.sum()} weights, max rel {rel.max():.2e}", flush=True)
    sys.stdout.flush()
    assert np.array_equal(fg, fo) and np.all(Wg[~ok] == 0)
    assert ok.any() and rel.max() <= RTOL


@pytest.mark.parametrize("name", sorted(RES_CASES))
def test_folded_nodes_fp32_amplitude(name):
    """The FP32-amplitude resonance nodes on folded kinematics, against the FP64 oracle.
    Bound: an FP32 rounding is 6e-8, a node runs some tens of them on its largest terms,
    and the screened amplitude can be 1/10 of its parts, squared: 6e-8 x 50 x 20 = 6e-5,
    on the weights that FP32 resolves (above 1e-8 of the largest)."""
    over, change = RES_CASES[name]
    cfg = small_tables(abi.cfg_default(7), 500)
    for key, value in over.items():
        setattr(cfg, key, value)
    if change:
        change(cfg)
    ref = abi.GraCfg.from_buffer_copy(cfg)
    cfg.amp_precision, ref.amp_precision = abi.GRA_AMP_FP32, abi.GRA_AMP_FP64
    print(f"case: {name}, FP32 amplitude, 65 points", flush=True)
    u = np.random.default_rng(72).random((65, cfg.dim))
    with MContinuum(cfg) as P:
        Wg, _, fg = P.eval(u)
    Wo, _, fo = ol.OracleRun(ref).eval(u)
    big = Wo > 1e-8 * Wo.max()
    rel = np.abs(Wg[big] - Wo[big]) / Wo[big]
    print(f"{big.sum()} weights, max rel {rel.max():.2e}", flush=True)
    assert np.array_equal(fg, fo) and rel.max() <= 6e-5
