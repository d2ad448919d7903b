"""Performance cases: what a user of this package has the GPU do.

A case names a process (one of the preset workloads of gra_hip_cfg_default, with
its amplitude precision), a call and a size:

  setup           create a screened process (its eikonal tables) and read the tables
  weights         batched EventWeight on host arrays (MContinuum.eval)
  weights_device  batched EventWeight on device buffers
  integrate       one VEGAS pass on an adapted grid (accumulators of the iteration)
  generate        one hit-or-miss generation pass on an adapted grid, events in
                  pinned host memory
  flow_train      one Adam step of the flow sampler
  flow_sample     one sampling pass of the flow sampler

prepare() makes the handle, the grid, max f and the flow that a program holds when
it makes such a call. The grid is adapted on the unscreened process: screening is a
smooth factor of order one, so the grid is the one a run meets, and it costs little.
"""
import ctypes as C
import math

import numpy as np
import torch

from graniitti_amd import abi
from graniitti_amd.process import MContinuum, MGraniitti, vegas_cfg

# process: (preset, unscreened preset of the same phase space, amplitude precision,
# largest size of the drawn cases)
PROCESSES = {
    "pipi": (1, 1, abi.GRA_AMP_FP64, 1 << 20),
    "pipi_screened": (2, 1, abi.GRA_AMP_FP32, 1 << 20),
    "pipi_screened_fp64": (2, 1, abi.GRA_AMP_FP64, 1 << 18),
    "pipi_gauss": (11, 1, abi.GRA_AMP_FP32, 1 << 20),
    "pipi_factorized": (4, 4, abi.GRA_AMP_FP64, 1 << 20),
    "pipi_factorized_screened": (5, 4, abi.GRA_AMP_FP32, 1 << 20),
    "rhorho_screened": (3, 3, abi.GRA_AMP_FP32, 1 << 18),
    "rhorho_screened_fp64": (3, 3, abi.GRA_AMP_FP64, 1 << 16),
    "resonances": (6, 6, abi.GRA_AMP_FP64, 1 << 20),
    "resonances_screened": (7, 6, abi.GRA_AMP_FP64, 1 << 16),
    "resonances_screened_fp32": (7, 6, abi.GRA_AMP_FP32, 1 << 17),
    "tensor_pipi": (9, 9, abi.GRA_AMP_FP64, 1 << 20),
    "tensor_pipi_screened": (10, 9, abi.GRA_AMP_FP64, 1 << 17),
}
# flow: layers, spline bins, hidden width, hidden layers
FLOWS = {"small": (4, 8, 64, 2), "pipi": (6, 16, 128, 2), "rhorho": (10, 32, 256, 3)}


def listed():
    return [
        # one EventWeight call of a program that walks the phase space by itself: latency
        {"name": "weights_one_point", "call": "weights", "process": "pipi", "n": 1},
        # a ragged batch of caller's points, host arrays in and out
        {"name": "weights_screened_4999", "call": "weights", "process": "pipi_screened",
         "n": 4999},
        # the reference-order FP64 amplitude, for validation and for reweighting
        {"name": "weights_screened_fp64", "call": "weights_device",
         "process": "pipi_screened_fp64", "n": 100003},
        # starting a screened run: both eikonal tables
        {"name": "setup_screened", "call": "setup", "process": "pipi_screened", "n": 1},
        # integration of the unscreened continuum (bench.py's pass size)
        {"name": "integrate_pipi", "call": "integrate", "process": "pipi", "n": 1 << 20},
        # integration of the screened continuum, the flagship process
        {"name": "integrate_screened", "call": "integrate", "process": "pipi_screened",
         "n": 1 << 20},
        # event generation, bench.py's timed step
        {"name": "generate_screened", "call": "generate", "process": "pipi_screened",
         "n": 1 << 20},
        # integration of the screened rho rho pair (tensor pomeron, nine helicity amplitudes)
        {"name": "integrate_rhorho", "call": "integrate", "process": "rhorho_screened",
         "n": 1 << 18},
        # integration of continuum + resonances, FP64 loop nodes
        {"name": "integrate_resonances", "call": "integrate", "process": "resonances_screened",
         "n": 1 << 16},
        # generation of continuum + resonances, FP32-amplitude loop nodes
        {"name": "generate_resonances_fp32", "call": "generate",
         "process": "resonances_screened_fp32", "n": 1 << 17},
        # training of the flow sampler (bench.py's flow and batch)
        {"name": "flow_train_pipi", "call": "flow_train", "process": "pipi_screened",
         "n": 1 << 18, "flow": "pipi"},
        # sampling pass of the large flow on the screened rho rho pair
        {"name": "flow_sample_rhorho", "call": "flow_sample", "process": "rhorho_screened",
         "n": 100000, "flow": "rhorho"},
    ]


def draw(rng):
    call = rng.choice(["weights", "weights_device", "integrate", "generate", "weights",
                       "weights_device", "integrate", "generate", "flow_train", "flow_sample"])
    if call.startswith("flow"):
        process = rng.choice(["pipi_screened", "rhorho_screened"])
        flow = rng.choice(["small", "pipi", "rhorho"])
        top = 1 << 16 if process == "rhorho_screened" or flow == "rhorho" else 1 << 18
        n = int(2.0 ** rng.uniform(10.0, math.log2(top)))
        if call == "flow_train":
            n = max(256, n // 256 * 256)
        return {"call": call, "process": process, "n": n, "flow": flow}
    process = rng.choice(sorted(PROCESSES))
    top = PROCESSES[process][3]
    if call == "weights":
        top = min(top, 1 << 16)
    n = int(2.0 ** rng.uniform(0.0 if call.startswith("weights") else 8.0, math.log2(top)))
    return {"call": call, "process": process, "n": max(1, n)}


def _config(process):
    preset, _, precision, _ = PROCESSES[process]
    cfg = abi.cfg_default(preset)
    cfg.amp_precision = precision
    return cfg


def _adapted_grid(process, seed):
    """A grid after three VEGAS iterations of the unscreened process."""
    cfg = abi.cfg_default(PROCESSES[process][1])
    cfg.screening = 0
    cfg.amp_precision = abi.GRA_AMP_FP64
    with MContinuum(cfg) as P:
        G = MGraniitti(P)
        G.Integrate(vegas_cfg(1 << 17, 1, burnin=3, seed=seed + 1))
        return abi.GraGrid.from_buffer_copy(G.grid)


class _Records:
    """The records of a PinnedEvents buffer as an array that keeps the buffer."""

    def __init__(self, events):
        self.events = events
        self.__array_interface__ = np.ctypeslib.as_array(events.buf).__array_interface__


def prepare(case, seed):
    call, n = case["call"], case["n"]
    cfg = _config(case["process"])
    state = {"call": call, "n": n, "cfg": cfg, "seed": seed}
    if call == "setup":
        # other beam energies, other tables
        cfg.beam_E1 = cfg.beam_E2 = 3500.0 + 500.0 * (seed % 15)
        return state
    P = state["P"] = MContinuum(cfg)
    if call == "weights":
        state["u"] = np.random.default_rng(seed).random((n, cfg.dim))
        return state
    if call == "weights_device":
        g = torch.Generator(device="cuda").manual_seed(seed)
        state["u"] = torch.rand(n, cfg.dim, dtype=torch.float64, device="cuda", generator=g)
        state["W"] = torch.empty(n, dtype=torch.float64, device="cuda")
        state["amp2"] = torch.empty(n, dtype=torch.float64, device="cuda")
        state["flags"] = torch.empty(n, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()  # the handle works on a stream of its own
        return state
    state["grid"] = _adapted_grid(case["process"], seed)
    if call == "integrate":
        # the iteration's first pass allocates the handle's buffers, as in a run
        P.vegas_iterate(state["grid"], 256, seed, 0)
    elif call == "generate":
        state["maxf"] = P.vegas_iterate(state["grid"], 1 << 14, seed, 7).maxf
        # room for every event of a pass (a few percent of the points are accepted)
        state["events"] = abi.PinnedEvents(n // 16 + 64)
        C.memset(state["events"].buf, 0, C.sizeof(state["events"].buf))
        state["records"] = np.asarray(_Records(state["events"]))
    else:
        L, K, H, depth = FLOWS[case["flow"]]
        fc = abi.GraFlowCfg()
        fc.dim, fc.layers, fc.bins, fc.hidden, fc.depth = cfg.dim, L, K, H, depth
        fc.batch, fc.lr, fc.beta1, fc.beta2, fc.eps = 1 << 17, 1e-3, 0.9, 0.999, 1e-8
        fc.seed, fc.ess_fallback = seed + 2, 0.1
        if call == "flow_train":
            fc.batch = n
        abi.check(P.lib.gra_hip_flow_init(P.h, C.byref(fc)), P.h)
        abi.check(P.lib.gra_hip_flow_set_grid(P.h, C.byref(state["grid"])), P.h)
        abi.check(P.lib.gra_hip_flow_train(P.h, 3, None), P.h)  # no longer the identity
        count = C.c_uint64()
        abi.check(P.lib.gra_hip_flow_param_count(P.h, C.byref(count)), P.h)
        state["theta"] = np.empty(count.value, dtype=np.float32)
        state["w"], state["x"] = np.empty(n), np.empty((n, cfg.dim))
    return state


def _flow_stats(s):
    return {"sigma": s.sigma, "sigma_err": s.sigma_err, "cv2": s.cv2, "ess": s.ess,
            "maxw": s.maxw}


def run(state):
    call, n, seed = state["call"], state["n"], state["seed"]
    if call == "setup":
        with MContinuum(state["cfg"]) as P:
            node, mbt, msa = P.eikonal_tables()
        return {"node": node, "mbt": mbt, "msa": msa}
    P = state["P"]
    if call == "weights":
        W, amp2, flags = P.eval(state["u"])
        return {"W": W, "amp2": amp2, "flags": flags}
    if call == "weights_device":
        abi.check(P.lib.gra_hip_eval_points_device(
            P.h, state["u"].data_ptr(), n, state["W"].data_ptr(), state["amp2"].data_ptr(),
            state["flags"].data_ptr()), P.h)
        return {"W": state["W"], "amp2": state["amp2"], "flags": state["flags"]}
    if call == "integrate":
        st = P.vegas_iterate(state["grid"], n, seed, 1)
        D = state["cfg"].dim * abi.GRA_VEGAS_BINS
        return {"fsum": st.fsum, "f2sum": st.f2sum, "maxW": st.maxW, "maxf": st.maxf,
                "n_valid": st.n_valid, "n_fid_ok": st.n_fid_ok, "n_kin_ok": st.n_kin_ok,
                "fmat": np.array(st.fmat[:D]), "f2mat": np.array(st.f2mat[:D])}
    if call == "generate":
        st, ev = abi.GraGenStats(), state["events"]
        abi.check(P.lib.gra_hip_generate(P.h, C.byref(state["grid"]), n, seed, 1, state["maxf"],
                                         ev.buf, ev.n, C.byref(st)), P.h)
        a = state["records"]  # the first st.stored of them hold the events
        return {"p": a["p"], "f": a["f"], "index": a["index"].view(np.int64), "n_p": a["n_p"],
                "trials": st.trials, "valid": st.valid, "accepted": st.accepted,
                "overflow": st.overflow, "stored": st.stored}
    s = abi.GraFlowStats()
    if call == "flow_train":
        abi.check(P.lib.gra_hip_flow_train(P.h, 1, C.byref(s)), P.h)
        abi.check(P.lib.gra_hip_flow_get_params(P.h, abi.fptr(state["theta"])), P.h)
        return {"theta": state["theta"], **_flow_stats(s)}
    abi.check(P.lib.gra_hip_flow_sample(P.h, n, seed, abi.dptr(state["w"]), abi.dptr(state["x"]),
                                        C.byref(s)), P.h)
    return {"w": state["w"], "x": state["x"], **_flow_stats(s)}


# Operations of one point without its loop, and of one loop node, as the cheapest
# known formulation needs them (the FP32 continuum node is counted by the library's
# op-counting build: 138; the others by hand)
_TREE_FLOPS = 1500
_NODE_FLOPS = {2: 138, 5: 138, 11: 138, 3: 1300, 7: 900, 10: 350}


def work(case):
    call, n = case["call"], case["n"]
    cfg = _config(case["process"])
    if call == "setup":
        rows = cfg.n_bt + cfg.n_kt2 + 2
        return {"bytes": rows * 24.0, "flops": rows * (cfg.n_fb + 1) * 30.0}
    flops = float(_TREE_FLOPS)
    if cfg.screening:
        nodes = (cfg.n_loop_phi + 1) * (cfg.n_loop_kt + 1)
        # points that pass the cuts: about 3 of 4 on an adapted grid, 1 of 20 uniform
        share = 0.05 if call.startswith("weights") else 0.75
        flops += share * nodes * _NODE_FLOPS[PROCESSES[case["process"]][0]]
    nbytes = 0.0
    if call.startswith("weights"):
        nbytes = cfg.dim * 8.0 + 17.0
    elif call == "flow_sample":
        nbytes = cfg.dim * 8.0 + 8.0
    elif call != "flow_train":
        nbytes = 16.0 / n * cfg.dim * abi.GRA_VEGAS_BINS
    if call.startswith("flow"):
        L, K, H, depth = FLOWS[case["flow"]]
        half = cfg.dim / 2.0
        weights = L * (half * H + (depth - 1) * H * H + H * half * (3 * K - 1))
        # forward; training adds the density direction and its two backward products
        flops += 2.0 * weights * (4.0 if call == "flow_train" else 1.0)
        nbytes += 4.0 * weights * (7.0 if call == "flow_train" else 1.0) / n
    return {"bytes": nbytes * n, "flops": flops * n}


# ---------------------------------------------------------------------------
# exact(): the Regge continuum PP[CON]<C> in float64, from its textbook form
# ---------------------------------------------------------------------------
_F64 = {"dtype": torch.float64, "device": "cuda"}
_MP, _MPI = 0.938272081, 0.13957061
_RAP, _KT_MAX, _PT_MAX, _PT_EPS = 0.9, 5.0, 2.5, 1e-12
_A0, _AP, _GN, _FC1, _FC2, _FC3, _B_POW, _C_PI = 1.088, 0.20, 8.20, 0.34, 5.0, 10.0, 0.5, 35.00184
_HBARC = 6.582119514e-25 * 2.99792458e8


def _eta(alpha):
    """Regge signature factor of positive signature"""
    phase = torch.exp(-1j * math.pi * alpha)
    return -(1.0 + phase) / torch.sin(math.pi * alpha)


def _simpson(n):
    w = torch.ones(n + 1, **_F64)
    w[1:n:2], w[2:n:2] = 4.0, 2.0
    return w / 3.0


def _bessel_sum(x, q, f):
    """sum_q f_q J0(x q) for every x"""
    out = torch.empty(len(x), dtype=torch.complex128, device="cuda")
    for k in range(0, len(x), 1024):
        j0 = torch.special.bessel_j0(x[k:k + 1024, None] * q[None, :])
        out[k:k + 1024] = torch.complex(j0 @ f.real, j0 @ f.imag)
    return out


def _eikonal(E, n=10000):
    """Density and screening-amplitude tables (x, value) of the soft pomeron"""
    s = 4.0 * E * E
    kt = 1e-9 + (30.0 - 1e-9) / n * torch.arange(n + 1, **_F64)
    t = -kt * kt
    mpi = 0.13957018
    tau = 4.0 * mpi * mpi / torch.abs(t)
    rt = torch.sqrt(1.0 + tau)
    loop = (4.0 / tau) / (1.0 - t / _FC3) ** 2 * (
        2.0 * tau - (1.0 + tau) ** 1.5 * torch.log((rt + 1.0) / (rt - 1.0))
        + math.log(1.0 / mpi ** 2))
    alpha = 1.0 + 0.098 + 0.065 * t - (2.0 / 3.0 * _GN) ** 2 * mpi ** 2 / (
        32.0 * math.pi ** 3) * loop
    form = 1.0 / ((1.0 - t / _FC1) * (1.0 - t / _FC2))
    amp = _eta(alpha) * (_GN * form) ** 2 * s ** alpha
    h = float(kt[1] - kt[0])
    b = 1e-6 + (10.0 / (_HBARC * 1e15) - 1e-6) / n * torch.arange(n + 1, **_F64)
    omega = _bessel_sum(b, kt, amp * kt * _simpson(n) * h) / (2.0 * math.pi * s)
    profile = 1j * (1.0 - torch.exp(0.5j * omega))
    h = float(b[1] - b[0])
    k2 = 1e-6 + (25.0 - 1e-6) / n * torch.arange(n + 1, **_F64)
    aeik = _bessel_sum(torch.sqrt(k2), b, profile * b * _simpson(n) * h) * (4.0 * math.pi * s)
    return b, omega, k2, aeik


def _loop_nodes(E):
    """(kx, ky, weight kt A_eik) of the 16 x 31 Simpson 3/8 loop grid"""
    _, _, k2, aeik = _eikonal(E)
    kt = 1e-4 + (3.0 - 1e-4) / 30 * torch.arange(31, **_F64)
    i = torch.clamp(((kt * kt - 1e-6) / (k2[1] - k2[0])).long(), 0, len(k2) - 2)
    a = aeik[i] + (aeik[i + 1] - aeik[i]) * ((kt * kt - k2[i]) / (k2[i + 1] - k2[i]))
    phi = 2.0 * math.pi / 15 * torch.arange(16, **_F64)

    def simpson38(m):
        w = torch.full((m + 1,), 3.0, **_F64)
        w[0::3], w[0], w[m] = 2.0, 1.0, 1.0
        return w

    w = simpson38(15)[:, None] * simpson38(30)[None, :] * kt[None, :] * a[None, :]
    w = w * (9.0 * (2.0 * math.pi / 15) * float(kt[1] - kt[0]) / 64.0)
    return ((torch.cos(phi)[:, None] * kt).reshape(-1), (torch.sin(phi)[:, None] * kt).reshape(-1),
            w.reshape(-1), a)


def _proton_z(rs, m, pt1, pt2, E5, pz5):
    """Longitudinal momentum of proton 1 from energy and momentum conservation"""
    e, p = rs - E5, -pz5
    m1, m2, M2 = m * m + pt1, m * m + pt2, (rs - E5) ** 2 - pz5 ** 2
    a = 0.5 * (M2 + m1 - m2)
    return (a * p + e * torch.sqrt(a * a - m1 * M2)) / M2


def _amplitude(E, p1, p2, c3, c4):
    """Regge amplitude of the proton momenta p1, p2 with the central pair c3, c4
    (tuples E, x, y, z), and t1, t2"""
    pz = math.sqrt(E * E - _MP * _MP)

    def sq(v):
        return v[0] ** 2 - v[1] ** 2 - v[2] ** 2 - v[3] ** 2

    def add(a, b):
        return tuple(x + y for x, y in zip(a, b))

    q1 = (E - p1[0], -p1[1], -p1[2], pz - p1[3])
    t1, t2 = sq(q1), sq((E - p2[0], -p2[1], -p2[2], -pz - p2[3]))
    form = [_GN / ((1.0 - t / _FC1) * (1.0 - t / _FC2)) for t in (t1, t2)]
    e1, e2 = _A0 + _AP * t1, _A0 + _AP * t2
    total = 0.0
    for a, b in ((c3, c4), (c4, c3)):
        off = sq(tuple(x - y for x, y in zip(q1, a))) - _MPI ** 2
        ff = 1.0 / (1.0 - off / _B_POW)
        total = total + sq(add(p1, a)) ** e1 * sq(add(p2, b)) ** e2 * ff ** 2 / off
    eta0 = _eta(torch.tensor(_A0, dtype=torch.complex128, device="cuda"))
    phase = torch.exp(-0.5j * math.pi * _AP * (t1 + t2))
    return eta0 ** 2 * phase * (form[0] * form[1] * (_C_PI / _GN) ** 2 * total), t1, t2


def _weights(x, screened, E=6500.0):
    """Event weight (barn) and |M|^2 at the points x (n, 8) of the hypercube"""
    if screened:
        kx, ky, cn, _ = _loop_nodes(E)
    W, A2 = torch.zeros(len(x), **_F64), torch.zeros(len(x), **_F64)
    rs = 2.0 * E
    s, l0, l1 = rs * rs, math.log(_PT_EPS), math.log(_PT_MAX)
    pt = torch.exp(l0 + (l1 - l0) * x[:, :2])
    phi = 2.0 * math.pi * x[:, 2:4]
    px, py = pt * torch.cos(phi), pt * torch.sin(phi)
    kt, kphi = _KT_MAX * x[:, 4], 2.0 * math.pi * x[:, 5]
    y = -_RAP + 2.0 * _RAP * x[:, 6:8]
    central = []
    for sign, rap in ((1.0, y[:, 0]), (-1.0, y[:, 1])):
        cx = 0.5 * (sign * kt * torch.cos(kphi) - px[:, 0] - px[:, 1])
        cy = 0.5 * (sign * kt * torch.sin(kphi) - py[:, 0] - py[:, 1])
        mt = torch.sqrt(_MPI ** 2 + cx * cx + cy * cy)
        central.append((mt * torch.cosh(rap), cx, cy, mt * torch.sinh(rap)))
    c3, c4 = central

    def protons(dx, dy, at):
        ax, ay = px[at, 0, None] - dx, py[at, 0, None] - dy
        bx, by = px[at, 1, None] + dx, py[at, 1, None] + dy
        E5, z5 = (c3[0] + c4[0])[at, None], (c3[3] + c4[3])[at, None]
        az = _proton_z(rs, _MP, ax * ax + ay * ay, bx * bx + by * by, E5, z5)
        bz = -z5 - az
        return ((torch.sqrt(_MP ** 2 + ax * ax + ay * ay + az * az), ax, ay, az),
                (torch.sqrt(_MP ** 2 + bx * bx + by * by + bz * bz), bx, by, bz))

    ok = torch.ones(len(x), dtype=torch.bool, device="cuda")
    for c in (c3, c4):
        p = torch.sqrt(c[1] ** 2 + c[2] ** 2 + c[3] ** 2)
        eta = 0.5 * torch.log((p + c[3]) / (p - c[3]))
        ok &= (torch.hypot(c[1], c[2]) >= 0.15) & (torch.abs(eta) <= 0.9)
    zero = torch.zeros(1, **_F64)
    step = (1 << 22) // (len(kx) if screened else 1)
    where = torch.nonzero(ok)[:, 0]
    for k in range(0, len(where), step):
        at = where[k:k + step]
        c = [tuple(v[at, None] for v in u) for u in (c3, c4)]
        p1, p2 = protons(zero, zero, at)
        amp = _amplitude(E, p1, p2, *c)[0]
        if screened:
            q1, q2 = protons(kx[None, :], ky[None, :], at)
            a, t1, t2 = _amplitude(E, q1, q2, *c)
            a = torch.where((t1 <= 0) & (t2 <= 0), a, torch.zeros_like(a))
            amp = amp[:, 0] + 1j / (8.0 * math.pi ** 2 * s) * (a @ cn)
        amp2 = torch.abs(amp).reshape(-1) ** 2
        z1, z2 = p1[3][:, 0] / p1[0][:, 0], p2[3][:, 0] / p2[0][:, 0]
        pp = pt[at, 0] * pt[at, 1]
        psw = pp / (4.0 * p1[0][:, 0] * p2[0][:, 0]) / torch.abs(z1 - z2) * kt[at]
        psw = psw / (16.0 * (2.0 * math.pi) ** 8)
        vol = _KT_MAX * (2.0 * math.pi) ** 3 * (2.0 * _RAP) ** 2 * (l1 - l0) ** 2 * pp
        W[at] = psw * vol * amp2 * (_HBARC ** 2 * 1e28) / (2.0 * s)
        A2[at] = amp2
    return W, A2


def _uniforms(seed, iteration, n, dim):
    """The counter-based (Philox4x32-10) uniforms of the points 0 .. n - 1"""
    index, mask = torch.arange(n, device="cuda"), 0xFFFFFFFF
    u = torch.empty(n, dim, **_F64)
    for b in range((dim + 1) // 2):
        c = [torch.full_like(index, b), index & mask, index >> 32,
             torch.full_like(index, iteration)]
        k0, k1 = seed & mask, (seed >> 32) & mask
        for _ in range(10):
            p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
            c = [((p1 >> 32) & mask) ^ c[1] ^ k0, p1 & mask,
                 ((p0 >> 32) & mask) ^ c[3] ^ k1, p0 & mask]
            k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
        u[:, 2 * b] = ((c[0] << 21) | (c[1] >> 11)).double() * 2.0 ** -53
        if 2 * b + 1 < dim:
            u[:, 2 * b + 1] = ((c[2] << 21) | (c[3] >> 11)).double() * 2.0 ** -53
    return u


def exact(case, seed):
    """Float64 values of the Regge continuum's outputs; None for the processes whose
    amplitudes (resonances, tensor pomeron), phase space (<F>) or quadrature are not
    restated here, for the flow's and the generation's outputs, and for counts."""
    call, process = case["call"], case["process"]
    if process not in ("pipi", "pipi_screened", "pipi_screened_fp64"):
        return None
    screened = process != "pipi"
    if call == "setup":
        E = 3500.0 + 500.0 * (seed % 15)
        b, omega, k2, aeik = _eikonal(E)
        _, _, _, node = _loop_nodes(E)
        return {"node": node, "mbt": torch.stack([b, omega.real, omega.imag], 1),
                "msa": torch.stack([k2, aeik.real, aeik.imag], 1)}
    if call in ("weights", "weights_device"):
        u = prepare(case, seed)["u"]
        W, amp2 = _weights(torch.as_tensor(u, **_F64), screened)
        return {"W": W, "amp2": amp2, "flags": None}
    if call == "integrate":
        st = prepare(case, seed)
        D, B = st["cfg"].dim, abi.GRA_VEGAS_BINS
        edges = torch.zeros(D, B + 1, **_F64)
        edges[:, 1:] = torch.as_tensor(abi.grid_xmat(st["grid"]).copy(), **_F64)
        u = _uniforms(seed, 1, case["n"], D)
        bins = torch.clamp((u * B).long(), max=B - 1)
        x, vw = torch.empty_like(u), torch.ones(len(u), **_F64)
        for j in range(D):
            lo, hi = edges[j][bins[:, j]], edges[j][bins[:, j] + 1]
            x[:, j] = lo + (u[:, j] * B - bins[:, j]) * (hi - lo)
            vw = vw * ((hi - lo) * B)
        W, _ = _weights(x, screened)
        f = W * vw
        out = {"fsum": f.sum(), "f2sum": (f * f).sum(), "maxW": W.max(), "maxf": f.max(),
               "n_valid": None, "n_fid_ok": None, "n_kin_ok": None}
        for name, v in (("fmat", f), ("f2mat", f * f)):
            h = torch.zeros(D, B, **_F64)
            for j in range(D):
                h[j] = torch.bincount(bins[:, j], weights=v, minlength=B)
            out[name] = h.reshape(-1)
        return out
    return None
