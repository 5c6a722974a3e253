"""The framework's everyday calls, as timing cases.

A case is a dict of plain values; `listed()` holds the fixed ones and
`draw(rng)` gives more of the same ranges.  `prepare(case, seed)` builds what
a program has in hand before the call, `run(state)` makes one pass through
the public entry points and returns the pass's results, `work(case)` counts
the bytes and operations a pass cannot do without and `exact(case, seed)`
computes the results in plain numpy FP64.

Kinds of case:
  law       the point-wise law on host arrays (sma160_eval): one element's 8
            Gauss points is the call the Fortran drop-in makes per element;
            tens of thousands of points is a vectorised element loop
  law_dev   the same law on arrays that already live on the GPU
  bar, cantilever, specimens, tube
            one output interval of an explicit run: `steps` steps, then the
            fields the program writes out (displacement and velocity, or all
            that a restart needs).  In FP32 mode the program keeps its output
            in single precision, the precision of that mode's forces.
  mlp_infer, mlp_train
            inference of the surrogate network, and mini-batches of its
            training followed by reading the parameters back
"""
import math
import os

import numpy as np
import torch

import alya_sma_amd
from alya_sma_amd import problems
from alya_sma_amd._lib import check, lib
from alya_sma_amd.solid import (Solidz, eval_sld_stress_model_160,
                                eval_sld_stress_model_160_device)
from alya_sma_amd.surrogate import LOSS_WEIGHTS, WEIGHTS, Surrogate

# operations per Gauss point and step (add, mul, div) of the law and the
# element loop, and per node and step of the integrator (oracle/flops_per_gp.txt)
GP_FLOPS = {"kinematics": 544.0, "sma": 612.0, "neo": 136.0, "force": 354.0}
LAW_FLOPS = 612.0 + 90.0
NODE_FLOPS = 34.5
MLP_FLOPS = 2 * 52736
DAMPED = (1.0e5, 0.0)          # Rayleigh (alpha, beta) of the cantilever deck


def listed():
    return [
        # the Fortran drop-in's call: one element's Gauss points, host arrays
        dict(name="law_element", kind="law", n=8, mats=1),
        # a vectorised element loop's points on host arrays, many materials
        dict(name="law_host", kind="law", n=40001, mats=64),
        # points of the 400x20x20 cantilever, resident on the GPU
        dict(name="law_device", kind="law_dev", n=1280000, mats=256),
        # the uniaxial bar of the reference test: launch-bound, full restart
        dict(name="bar_fp64", kind="bar", nx=10, ny=2, nz=2, steps=200, mode=0, scheme=0,
             restart=True),
        # the headline cantilever in both precisions
        dict(name="cantilever_fp64", kind="cantilever", nx=400, ny=20, nz=20, steps=100, mode=0,
             scheme=0, damped=False, restart=False),
        dict(name="cantilever_fp32", kind="cantilever", nx=400, ny=20, nz=20, steps=100, mode=1,
             scheme=0, damped=False, restart=False),
        # a ragged mid-size mesh with the reference decks' integrator
        # (Tchamwa-Wielgosz), Rayleigh damping and gravity, full restart
        dict(name="cantilever_damped", kind="cantilever", nx=41, ny=9, nz=7, steps=75, mode=0,
             scheme=1, damped=True, restart=True),
        # many uneven specimens stepped as one mesh, own material rows
        dict(name="specimens_fp64", kind="specimens", n=64, mesh_seed=3, steps=50, mode=0,
             scheme=0, restart=False),
        # SMA tube in neo-Hookean tissue (curved elements, two laws)
        dict(name="tube_fp64", kind="tube", ntheta=180, nz=160, nr_tube=3, nr_tissue=21, steps=50,
             mode=0, scheme=0, restart=False),
        dict(name="tube_fp32", kind="tube", ntheta=180, nz=160, nr_tube=3, nr_tissue=21, steps=50,
             mode=1, scheme=0, restart=False),
        # the surrogate: its holdout set, and late-schedule mini-batches
        dict(name="mlp_infer", kind="mlp_infer", n=200000),
        dict(name="mlp_train", kind="mlp_train", batch=16384, batches=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["law", "law", "law_dev", "law_dev", "bar", "cantilever", "cantilever",
                       "cantilever", "specimens", "tube", "mlp_infer", "mlp_train"])
    if kind == "law":
        return dict(kind=kind, n=_log_int(rng, 8, 60000), mats=rng.choice([1, 1, 7, 64]))
    if kind == "law_dev":
        return dict(kind=kind, n=_log_int(rng, 500, 2000000), mats=rng.choice([1, 16, 256]))
    if kind == "mlp_infer":
        return dict(kind=kind, n=_log_int(rng, 500, 400000))
    if kind == "mlp_train":
        return dict(kind=kind, batch=_log_int(rng, 1000, 16384), batches=rng.choice([3, 5, 8]))
    case = dict(kind=kind, mode=rng.choice([0, 0, 1]), scheme=rng.choice([0, 0, 1]),
                steps=rng.randint(20, 50), restart=False)
    if kind == "bar":
        case.update(nx=rng.randint(4, 40), ny=rng.randint(1, 5), nz=rng.randint(1, 5),
                    steps=rng.randint(50, 200), restart=True)
    elif kind == "cantilever":
        case.update(nx=_log_int(rng, 20, 500), ny=_log_int(rng, 3, 24), nz=_log_int(rng, 3, 24),
                    steps=rng.randint(30, 100), damped=rng.random() < 0.25)
    elif kind == "specimens":
        case.update(n=rng.randint(3, 56), mesh_seed=rng.randint(1, 1000))
    else:
        case.update(ntheta=_log_int(rng, 36, 180), nz=_log_int(rng, 20, 160),
                    nr_tube=rng.randint(1, 4), nr_tissue=_log_int(rng, 2, 20))
    return case


# ------------------------------------------------------------------ law points
def _law_points(case, seed, device):
    """Material rows, and per point: material, Young's modulus, deformation
    gradient (strains of 0.001 .. 0.02) and the history of the state one increment
    (a tenth of it) before."""
    n, nm = case["n"], case["mats"]
    r = np.random.default_rng([seed, 1])
    props = np.tile(problems.NITINOL, (nm, 1))
    props[:, [0, 3, 4, 9, 10]] *= r.uniform(0.9, 1.1, (nm, 5))
    if device == "cpu":
        t = lambda a: torch.from_numpy(a)
        normal = lambda *s: t(r.normal(size=s))
        uniform = lambda *s: t(r.uniform(size=s))
    else:
        g = torch.Generator(device=device).manual_seed(int(seed) * 2 + 1)
        t = lambda a: torch.from_numpy(a).to(device)
        normal = lambda *s: torch.randn(*s, generator=g, device=device, dtype=torch.float64)
        uniform = lambda *s: torch.rand(*s, generator=g, device=device, dtype=torch.float64)
    props = t(props)
    mat = torch.clamp((uniform(n) * nm).to(torch.int32), max=nm - 1)
    E = props[mat.long(), 0] * (1.0 + 0.02 * (2.0 * uniform(n) - 1.0))
    size = 0.001 + 0.019 * uniform(n)
    H = size * normal(9, n)
    H0 = H - 0.1 * size * normal(9, n)
    tr = (H0[0] + H0[4] + H0[8]) / 3.0
    en = torch.sqrt((H0[0] - tr) ** 2 + (H0[4] - tr) ** 2 + (H0[8] - tr) ** 2 +
                    0.5 * ((H0[1] + H0[3]) ** 2 + (H0[2] + H0[6]) ** 2 + (H0[5] + H0[7]) ** 2))
    p = props[mat.long()]
    # the law's answer to that state from rest
    G2, Rs, Rf = E / (1.0 + p[:, 1]), math.sqrt(2.0 / 3.0) * p[:, 3], math.sqrt(2.0 / 3.0) * p[:, 4]
    xs = torch.where(G2 * en > Rs, G2 * en / (G2 * p[:, 2] + Rf), torch.zeros_like(en))
    f0 = G2 * (en - p[:, 2] * xs)
    xs = torch.clamp(xs, max=1.0)
    F = H
    F[[0, 4, 8]] += 1.0
    return props.contiguous(), mat, E, F.contiguous(), torch.stack([xs, f0, f0]).contiguous()


# ------------------------------------------------------------- explicit problems
def _ramp(m):
    return m * m * m * (10.0 - 15.0 * m + 6.0 * m * m)


def _problem(case, seed):
    """(problem, initial u, v, time): a run in progress, inside its load
    cycle, with part of the points past the transformation threshold."""
    r = np.random.default_rng([seed, 2])
    kind = case["kind"]
    if kind == "cantilever":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        h = 0.125
        lx, ly, lz = nx * h, ny * h, nz * h
        p = problems.cantilever_problem(nx, ny, nz, lx, ly, lz, seed=int(seed) + 1)
        x, y = p["coord"][:, 0], p["coord"][:, 1]
        # stretched and bent, most at the clamp
        e0, k0 = r.uniform(0.007, 0.010), 2.0 * r.uniform(0.002, 0.004) / lx
        s = 1.0 - x / lx
        u = np.zeros_like(p["coord"])
        u[:, 0] = e0 * (x - x * x / (2.0 * lx)) - k0 * lx / 3.0 * (1.0 - s ** 3) * (y - 0.5 * ly)
        u[:, 1] = k0 * (lx * x / 3.0 - lx * lx / 12.0 * (1.0 - s ** 4))
        v = np.zeros_like(u)
        v[:, 0] = r.uniform(-8.0e3, 8.0e3) * (x / lx)
        v[:, 2] = r.uniform(-4.0e3, 4.0e3) * (x / lx) ** 2
        if case["damped"]:
            p["damping"] = np.array([DAMPED])
            p["gravity"] = np.array([0.0, 0.0, -9810.0])
        return p, u, v, 0.05 * p["run"]["nsteps"] * p["run"]["dt"]
    if kind == "bar":
        p = problems.bar_problem(case["nx"], case["ny"], case["nz"], float(case["nx"]),
                                 float(case["ny"]), float(case["nz"]), nsteps=20000)
        t_half = 0.5 * p["run"]["nsteps"] * p["run"]["dt"]
        amp = 0.06 * case["nx"] * np.array([0.0, 1.0, 0.0, 0.5, 0.0, 1.0, 0.0, 0.5, 0.0])
        tab = np.zeros((9, 4))
        tab[:, 0], tab[:, 3] = amp, t_half * np.arange(9)
        p["func_table"], p["func_npts"] = tab[None], np.array([9], np.int32)
        m = r.uniform(0.30, 0.36)
        e = 0.06 * _ramp(m)
        u = p["coord"] * np.array([e, -0.33 * e, -0.33 * e])
        return p, u, np.zeros_like(u), m * t_half
    if kind == "specimens":
        p = problems.batched_specimens(n=case["n"], seed=case["mesh_seed"], nsteps=20000)
        t_half = 0.5 * p["run"]["nsteps"] * p["run"]["dt"]
        m = r.uniform(0.30, 0.36)
        spec = np.zeros(p["coord"].shape[0], np.int64)
        spec[p["lnods"]] = p["mat_of_elem"][:, None]
        e = p["specimens"]["amplitude"][spec] * _ramp(m)
        c = p["coord"] - np.stack([0 * e, 2.0 * spec, 0 * e], axis=1)
        u = c * np.stack([e, -0.33 * e, -0.33 * e], axis=1)
        return p, u, np.zeros_like(u), m * t_half
    p = problems.cylinder_problem(ntheta=case["ntheta"], nz=case["nz"], nr_tube=case["nr_tube"],
                                  nr_tissue=case["nr_tissue"], nsteps=40000)
    t_half = 0.5 * p["run"]["nsteps"] * p["run"]["dt"]
    m = r.uniform(0.24, 0.28)
    x, y = p["coord"][:, 0], p["coord"][:, 1]
    rad = np.hypot(x, y)
    ur = -0.4 * _ramp(m) * (10.0 - rad) / 6.0
    u = np.stack([ur * x / rad, ur * y / rad, 0 * x], axis=1)
    # crimped from both sides a little unevenly along the axis
    u[:, 2] = r.uniform(-2e-3, 2e-3) * p["coord"][:, 2] * (10.0 - rad) / 6.0
    return p, u, np.zeros_like(u), m * t_half


def _fields(case):
    return ("u", "v", "a", "sdv") if case["restart"] else ("u", "v")


# --------------------------------------------------------------------- surrogate
def _mlp_params(seed):
    """The committed network, perturbed a little."""
    d = np.load(os.path.join(os.path.dirname(os.path.abspath(alya_sma_amd.__file__)), "data",
                             os.path.basename(WEIGHTS)))
    r = np.random.default_rng([seed, 3])
    W, b = d["W"].astype(np.float32), d["b"].astype(np.float32)
    return (W * (1 + 0.02 * r.normal(size=W.size)).astype(np.float32),
            b * (1 + 0.02 * r.normal(size=b.size)).astype(np.float32))


def _mlp_samples(n, seed, device):
    """Features in their scaled ranges and targets that depend on them."""
    g = torch.Generator(device=device).manual_seed(int(seed) * 2)
    X = torch.randn(n, 16, generator=g, device=device)
    X[:, 4] = torch.rand(n, generator=g, device=device)                          # xS
    X[:, 7:15] = 2.0 * torch.rand(n, 8, generator=g, device=device) - 1.0        # T, material
    T = torch.tanh(X[:, :12] + 0.5 * X[:, 4:16]) + 0.1 * torch.randn(n, 12, generator=g, device=device)
    return X.contiguous(), T.contiguous()


def _adam_lr(case):
    return 1.0e-5                     # the end of the training schedule


# ----------------------------------------------------------------------- the API
def prepare(case, seed):
    kind = case["kind"]
    if kind == "law":
        props, mat, E, F, sdv = (a.numpy() for a in _law_points(case, seed, "cpu"))
        one = case["mats"] == 1
        return dict(kind=kind, props=props, F=F, sdv=sdv, mat=None if one else mat, E=None if one else E)
    if kind == "law_dev":
        props, mat, E, F, sdv = _law_points(case, seed, "cuda")
        n = case["n"]
        return dict(kind=kind, n=n, props=props, mat=mat, E=E, F=F, sdv=sdv,
                    out=torch.empty(3, n, dtype=torch.float64, device="cuda"),
                    S=torch.empty(9, n, dtype=torch.float64, device="cuda"),
                    flags=torch.empty(n, dtype=torch.int32, device="cuda"))
    if kind in ("mlp_infer", "mlp_train"):
        s = Surrogate()
        s.set_loss_weights(LOSS_WEIGHTS)
        s.set_params(*_mlp_params(seed))
        if kind == "mlp_infer":
            X, _ = _mlp_samples(case["n"], seed, "cuda")
            return dict(kind=kind, net=s, X=X, Y=torch.empty(case["n"], 12, device="cuda"))
        X, T = _mlp_samples(case["batch"] * case["batches"], seed, "cuda")
        return dict(kind=kind, net=s, X=X, T=T, batch=case["batch"], batches=case["batches"],
                    lr=_adam_lr(case))
    p, u, v, t = _problem(case, seed)
    dev = Solidz(p)
    dev.set_mode(case["mode"])
    dev.set("u", u)
    dev.set("v", v)
    dev.set("time", np.array([t]))
    return dict(kind=kind, dev=dev, dt=float(p["run"]["dt"]), steps=case["steps"],
                scheme=case["scheme"], mode=case["mode"], fields=_fields(case))


def run(state):
    kind = state["kind"]
    if kind == "law":
        return eval_sld_stress_model_160(state["props"], state["F"], state["sdv"],
                                         mat_of_gp=state["mat"], E_of_gp=state["E"])
    if kind == "law_dev":
        q = state
        eval_sld_stress_model_160_device(q["n"], q["props"].shape[0], q["props"].data_ptr(),
                                         q["F"].data_ptr(), q["sdv"].data_ptr(), q["out"].data_ptr(),
                                         q["S"].data_ptr(), flags_ptr=q["flags"].data_ptr(),
                                         mat_ptr=q["mat"].data_ptr(), E_ptr=q["E"].data_ptr())
        return q["out"], q["S"], q["flags"]
    if kind == "mlp_infer":
        X, Y = state["X"], state["Y"]
        check(lib().sma_mlp_forward_device(state["net"].h, X.shape[0], X.data_ptr(), Y.data_ptr(), None),
              "sma_mlp_forward_device")
        return Y
    if kind == "mlp_train":
        net, n, k = state["net"], state["batch"], state["batches"]
        x, t = state["X"].data_ptr(), state["T"].data_ptr()
        for j in range(k):
            loss = net.train_step(x + j * n * 64, t + j * n * 48, n, state["lr"], want_loss=j == k - 1)
        W, b = net.get_params()
        return dict(W=W, b=b, loss=loss)
    dev = state["dev"]
    dev.step(state["dt"], state["steps"], scheme=state["scheme"])
    out = {f: dev.get(f) for f in state["fields"]}
    if state["mode"] == 1:
        out = {f: a.astype(np.float32) for f, a in out.items()}
    return out


def _sizes(case):
    """(SMA elements, neo-Hookean elements, nodes) of an explicit case."""
    if case["kind"] in ("bar", "cantilever"):
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        return nx * ny * nz, 0, (nx + 1) * (ny + 1) * (nz + 1)
    if case["kind"] == "specimens":
        d = problems.batched_specimens(n=case["n"], seed=case["mesh_seed"])["specimens"]["dims"]
        return int(d.prod(axis=1).sum()), 0, int((d + 1).prod(axis=1).sum())
    ring = case["ntheta"] * case["nz"]
    nr = case["nr_tube"] + case["nr_tissue"]
    return case["nr_tube"] * ring, case["nr_tissue"] * ring, (nr + 1) * case["ntheta"] * (case["nz"] + 1)


def work(case):
    kind = case["kind"]
    if kind in ("law", "law_dev"):
        per = 72 + 24 + 24 + 72 + 4 + (0 if kind == "law" and case["mats"] == 1 else 12)
        return {"bytes": case["n"] * per + case["mats"] * 144, "flops": case["n"] * LAW_FLOPS}
    if kind == "mlp_infer":
        return {"bytes": case["n"] * 112 + 2 * 52736, "flops": case["n"] * MLP_FLOPS}
    if kind == "mlp_train":
        # samples read, master parameters and Adam moments read and written
        n = case["batch"] * case["batches"]
        return {"bytes": n * 112 + case["batches"] * 24 * 53260, "flops": 3 * n * MLP_FLOPS}
    sma, neo, nodes = _sizes(case)
    n = case["steps"]
    # per step: history read and written, connectivity and modulus; per node
    # the coordinates, u and v read and written, the mass; then the output
    per_step = sma * 8 * 53 + neo * 8 * 5 + nodes * (24 + 96 + 8)
    out = nodes * 24 * (3 if case["restart"] else 2) + (sma * 8 * 24 if case["restart"] else 0)
    f = GP_FLOPS["kinematics"] + GP_FLOPS["force"]
    flops = 8 * (sma * (f + GP_FLOPS["sma"]) + neo * (f + GP_FLOPS["neo"])) + nodes * NODE_FLOPS
    return {"bytes": n * per_step + out, "flops": n * flops}


# ------------------------------------------------------- plain FP64 counterparts
def _np_law(P, E, F, sdv):
    """The superelastic law at points: P [n, 18], E [n], F [n, 3, 3], sdv
    [3, n] -> (history [3, n], Kirchhoff stress [n, 3, 3])."""
    K, G = E / (3.0 - 6.0 * P[:, 1]), E / (2.0 + 2.0 * P[:, 1])
    eL, al = P[:, 2], P[:, 14]
    aux = math.sqrt(2.0 / 3.0) + al
    RfA, RsA = P[:, 4] * aux + P[:, 5] * P[:, 6], P[:, 3] * aux + P[:, 5] * P[:, 7]
    RfS, RsS = P[:, 10] * aux + P[:, 11] * P[:, 12], P[:, 9] * aux + P[:, 11] * P[:, 13]
    G1 = (2.0 * G + 9.0 * al * al * K) * eL
    H = F - np.eye(3)
    w, n = np.linalg.eigh(H + H.transpose(0, 2, 1) + H @ H.transpose(0, 2, 1))
    l = 0.5 * np.log1p(w)
    th = l.sum(1)
    e = l - th[:, None] / 3.0
    en = np.sqrt((e * e).sum(1))
    x0, fa0, fs0 = sdv
    load = lambda x: 2.0 * G * (en - eL * x) + 3.0 * al * K * (th - 3.0 * al * eL * x)
    fa = load(x0)
    fs = fa.copy()
    ka = (fa > fa0) & (fa - RsA > 0.0) & (x0 < 1.0)
    ks = (fs < fs0) & (fs - RsS < 0.0) & (x0 > 0.0)
    x = x0.copy()
    a, s = ka.astype(float), ks.astype(float)
    da, ds = np.zeros_like(x), np.zeros_like(x)
    ra = a * (fa - fa0) * (1.0 - x)
    rs = -s * (fs - fs0) * x
    live = (ka | ks) & (ra * ra + rs * rs > 1e-8)
    for _ in range(65):
        if not live.any():
            break
        j = np.nonzero(live)[0]
        ga = -G1[j] * da[j] - a[j] * ((fa - fa0)[j] + (1.0 - x[j]) * G1[j])
        gs = -G1[j] * ds[j] - s[j] * ((fs - fs0)[j] - x[j] * G1[j])
        m11, m12, m21, m22 = ga + (fa - RfA)[j], ga, gs, gs + (fs - RfS)[j]
        det = m11 * m22 - m12 * m21
        da[j] -= (m22 * ra[j] - m12 * rs[j]) / det
        ds[j] -= (m11 * rs[j] - m21 * ra[j]) / det
        x[j] += da[j] + ds[j]
        full = load(x)
        fa[j], fs[j] = full[j], full[j]
        ra[j] = (fa - RfA)[j] * da[j] + a[j] * (fa - fa0)[j] * (1.0 - x[j])
        rs[j] = (fs - RfS)[j] * ds[j] - s[j] * (fs - fs0)[j] * x[j]
        live[j] = np.sqrt(ra[j] ** 2 + rs[j] ** 2) > 1e-8
    x[live], fa[live], fs[live] = x0[live], fa0[live], fs0[live]
    x = np.clip(x, 0.0, 1.0)
    d = np.where(en[:, None] > np.finfo(float).eps, e / np.maximum(en, 1e-300)[:, None], 0.0)
    c = K * (th - 3.0 * al * eL * x)
    t = c[:, None] + 2.0 * G[:, None] * (e - (eL * x)[:, None] * d)
    return np.stack([x, fa, fs]), (n * t[:, None, :]) @ n.transpose(0, 2, 1)


def _np_neo(mu, K, F):
    J = np.linalg.det(F)
    b = F @ F.transpose(0, 2, 1)
    dev = b - np.trace(b, axis1=1, axis2=2)[:, None, None] / 3.0 * np.eye(3)
    return (mu * J ** (-2.0 / 3.0))[:, None, None] * dev + (J * K * (J - 1.0))[:, None, None] * np.eye(3)


def _np_table(tab, t):
    """Smooth load table: rows (vx, vy, vz, t) -> (vx, vy, vz) at t."""
    if t > tab[-1, 3]:
        return tab[-1, :3] * t / tab[-1, 3]
    for p, q in zip(tab[:-1], tab[1:]):
        if p[3] <= t <= q[3]:
            m = (t - p[3]) / (q[3] - p[3])
            return p[:3] + (q[:3] - p[:3]) * _ramp(m)
    return np.zeros(3)


def _np_run(case, seed):
    """The explicit run in numpy: (u, v, a, history) after `steps` steps."""
    p, u, v, t = _problem(case, seed)
    X, ln = p["coord"], p["lnods"].astype(np.int64)
    ne, npn = ln.shape[0], X.shape[0]
    sg = np.array([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1],
                   [-1, -1, 1], [1, -1, 1], [1, 1, 1], [-1, 1, 1]], float)
    c = 0.577350269189626
    gp = c * np.array([[x, y, z] for x in (-1, 1) for y in (-1, 1) for z in (-1, 1)], float)
    f = 1.0 + sg[None] * gp[:, None]                                   # [g, a, m]
    N = f.prod(2) / 8.0
    dN = np.stack([sg[None, :, 0] * f[:, :, 1] * f[:, :, 2], sg[None, :, 1] * f[:, :, 0] * f[:, :, 2],
                   sg[None, :, 2] * f[:, :, 0] * f[:, :, 1]], axis=2) / 8.0
    J = np.einsum("eai,gak->egik", X[ln], dN)
    dJ = np.linalg.det(J)
    dX = np.einsum("gak,egkj->egaj", dN, np.linalg.inv(J))              # dN_a/dX_j
    mat = p.get("mat_of_elem")
    mat = np.zeros(ne, np.int64) if mat is None else mat.astype(np.int64)
    P = p["props"][mat]
    E = p["E_of_elem"] if p.get("E_of_elem") is not None else P[:, 0]
    rho = p["rho"][mat]
    neo = np.zeros(ne, bool) if p.get("law_of_mat") is None else p["law_of_mat"][mat] == problems.LAW_NEOHOOKEAN
    sma8, neo8 = np.repeat(~neo, 8), np.repeat(neo, 8)
    P8, E8 = np.repeat(P, 8, axis=0), np.repeat(E, 8)
    add = lambda w: np.stack([np.bincount(ln.ravel(), w[..., d].ravel(), npn) for d in range(3)], axis=1)
    m = np.bincount(ln.ravel(), (rho[:, None] * np.einsum("eg,ga->ea", dJ, N)).ravel(), npn)
    fixed = ((p["fixmask"][:, None] >> np.arange(3)) & 1).astype(bool)
    fn, tabs = p.get("func_of_node"), p["func_table"]
    npts = p["func_npts"]
    a, sdv, dt, tw = np.zeros_like(u), np.zeros((3, ne * 8)), float(p["run"]["dt"]), case["scheme"] == 1
    for _ in range(case["steps"]):
        t += dt
        vel = v
        u, v = (u + dt * v + 1.033 * dt * dt * a, v + dt * a) if tw else (u + dt * (v + 0.5 * dt * a), v + 0.5 * dt * a)
        vals = np.stack([_np_table(tb[:k], t) for tb, k in zip(tabs, npts)] + [np.zeros(3)])
        u = np.where(fixed, vals[-1 if fn is None else fn], u)
        F = np.eye(3) + np.einsum("eai,egaj->egij", u[ln], dX)
        Fp = F.reshape(-1, 3, 3)
        tau = np.zeros_like(Fp)
        if sma8.any():
            sdv[:, sma8], tau[sma8] = _np_law(P8[sma8], E8[sma8], Fp[sma8], sdv[:, sma8])
        if neo8.any():
            tau[neo8] = _np_neo(P8[neo8, 0], P8[neo8, 1], Fp[neo8])
        PK = (tau @ np.linalg.inv(Fp).transpose(0, 2, 1)).reshape(F.shape) * dJ[..., None, None]
        r = -add(np.einsum("egij,egaj->eai", PK, dX))
        if p.get("damping") is not None:
            vg = np.einsum("ga,eai->egi", N, (v if tw else vel)[ln])
            w = p["damping"][mat, 0] * rho
            r -= add(np.einsum("e,eg,ga,egi->eai", w, dJ, N, vg))
        if p.get("fext0") is not None:
            r += _np_table(tabs[p["fext_func"]][:npts[p["fext_func"]]], t)[0] * p["fext0"]
        if p.get("gravity") is not None:
            r += m[:, None] * p["gravity"]
        a = r / m[:, None]
        if tw:
            v, a = np.where(fixed, 0.0, v), np.where(fixed, 0.0, a)
        else:
            v = v + 0.5 * dt * a
    return dict(u=u, v=v, a=a, sdv=sdv.T.reshape(ne, 8, 3))


def _np_layers(W, b):
    out, o, q = [], 0, 0
    for k, n in ((16, 128), (128, 128), (128, 128), (128, 128), (128, 12)):
        out.append([W[o:o + n * k].reshape(n, k).astype(np.float64), b[q:q + n].astype(np.float64)])
        o, q = o + n * k, q + n
    return out


def _np_forward(layers, X):
    """Pre-activations per layer and the inputs of each layer."""
    Z, Y = [], [X]
    for l, (W, b) in enumerate(layers):
        z = Y[-1] @ W.T + b
        Z.append(z)
        if l < 4:
            Y.append(z / (1.0 + np.exp(-z)))
    return Z, Y


def _np_train(case, seed):
    W, b = _mlp_params(seed)
    X, T = (q.double().cpu().numpy() for q in _mlp_samples(case["batch"] * case["batches"], seed, "cuda"))
    layers = _np_layers(W, b)
    mom = [[[np.zeros_like(p), np.zeros_like(p)] for p in l] for l in layers]
    n = case["batch"]
    for k in range(case["batches"]):
        Z, Y = _np_forward(layers, X[k * n:(k + 1) * n])
        d = Z[4] - T[k * n:(k + 1) * n]
        loss = float((LOSS_WEIGHTS * d * d).sum() / n)
        g = 2.0 * LOSS_WEIGHTS * d / n
        grads = [None] * 5
        for l in range(4, -1, -1):
            grads[l] = [g.T @ Y[l], g.sum(0)]
            if l:
                s = 1.0 / (1.0 + np.exp(-Z[l - 1]))
                g = (g @ layers[l][0]) * s * (1.0 + Z[l - 1] * (1.0 - s))
        for l in range(5):
            for q in range(2):
                mo = mom[l][q]
                mo[0] = 0.9 * mo[0] + 0.1 * grads[l][q]
                mo[1] = 0.999 * mo[1] + 0.001 * grads[l][q] ** 2
                layers[l][q] = layers[l][q] - _adam_lr(case) * (mo[0] / (1 - 0.9 ** (k + 1))) / (
                    np.sqrt(mo[1] / (1 - 0.999 ** (k + 1))) + 1e-8)
    return dict(W=np.concatenate([l[0].ravel() for l in layers]),
                b=np.concatenate([l[1] for l in layers]), loss=loss)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("law", "law_dev"):
        props, mat, E, F, sdv = (a.cpu().numpy() for a in
                                 _law_points(case, seed, "cpu" if kind == "law" else "cuda"))
        P = props[mat]
        if kind == "law" and case["mats"] == 1:
            E = P[:, 0]
        F = F.T.reshape(-1, 3, 3).transpose(0, 2, 1)
        new, tau = _np_law(P, E, F, sdv)
        Fi = np.linalg.inv(F)
        S = Fi @ tau @ Fi.transpose(0, 2, 1)
        return new, np.ascontiguousarray(S.transpose(0, 2, 1).reshape(-1, 9).T), None
    if kind == "mlp_infer":
        X, _ = _mlp_samples(case["n"], seed, "cuda")
        return _np_forward(_np_layers(*_mlp_params(seed)), X.double().cpu().numpy())[0][4]
    if kind == "mlp_train":
        return _np_train(case, seed)
    if kind != "specimens" and 8 * sum(_sizes(case)[:2]) * case["steps"] > 3.0e6:
        return None
    if kind == "specimens":
        return None        # more than a minute of numpy
    out = _np_run(case, seed)
    return {f: out[f] for f in _fields(case)}
