"""Measured cases: what a user of this framework has it do, through its public entry points.

A full-waveform-inversion program models shot records (AcousticPropagator, ElasticPropagator),
compares them with observed data (the misfits of adfwi_amd.fwi) and takes the gradient with
respect to the model (backward).  The listed cases are such calls over the range of sizes this
repository names: from one shot on the 100 x 200 grid of the small workload, where a pass is a
thousand tiny time steps, to 64 shots on the 384 x 1152 grid of the benchmark, where the state
does not fit any cache.  Both directions (modelling alone, modelling with its gradient), both
wave equations, PML and taper boundaries, 4th and 6th order, with and without a free surface,
one- and multi-component data, and grids that are no multiple of anything are among them.
The number of time steps is below the workloads' 1000-6000 where a pass would otherwise take
seconds; each step costs the same.

Models are layered gradients with smooth seeded heterogeneity.  Observed data are seeded
hyperbolic arrivals with the shots' own wavelet, so that no modelling run is needed for them.
All data are float32, the only type the propagators take.
"""
import math

import numpy as np
import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

DEV = "cuda:0"


def listed():
    ac = dict(wave="acoustic", nabc=20, dx=10.0, dt=1e-3, f0=10.0, fs=False)
    el = dict(wave="elastic", nabc=20, dx=5.0, dt=5e-4, f0=12.0, fs=True, order=4, abc="PML", source="mt", vti=False)
    return [
        # one shot on the small grid: a quick look at a model; 1000 steps of 34k points, all latency
        dict(ac, name="ac_model_1shot", nz=100, nx=200, shots=1, nt=1000, mode="model"),
        # the small workload of the benchmark's CPU baseline: one inversion iteration of ten shots
        dict(ac, name="ac_grad_10shots", nz=100, nx=200, shots=10, nt=1000, mode="grad", misfit="l2sq", par="vp", comp="p"),
        # one batch of the FWI driver on a marine model with a free surface and odd sizes: the
        # normalised waveform misfit
        dict(ac, name="ac_fwi_fs_odd", nz=89, nx=203, nabc=30, dx=40.0, dt=3e-3, f0=5.0, fs=True, shots=40, nt=1600,
             mode="grad", misfit="norm", par="vp", comp="p"),
        # a line of shots modelled for a survey design or a data set (no gradient)
        dict(ac, name="ac_model_16shots", nz=256, nx=768, shots=16, nt=1000, mode="model"),
        # two-parameter inversion of multi-component data (ocean-bottom nodes)
        dict(ac, name="ac_grad_rho_puw", nz=201, nx=401, shots=12, nt=700, mode="grad", misfit="l2sq", par="vp+rho",
             comp="puw"),
        # the benchmark's own workload with half its time steps: the largest call
        dict(ac, name="ac_grad_large", nz=384, nx=1152, nabc=40, dx=12.5, f0=8.0, shots=64, nt=2000, mode="grad",
             misfit="l2sq", par="vp", comp="p"),
        # one elastic shot on a small grid
        dict(el, name="el_model_1shot", nz=100, nx=200, shots=1, nt=1000, mode="model"),
        # the isotropic elastic workload: vertical-force shots, free surface, vx and vz data
        dict(el, name="el_grad_iso", nz=200, nx=600, nabc=40, f0=8.0, shots=32, nt=600, mode="grad", source="vf"),
        # the VTI workload: Thomsen parameters inverted too
        dict(el, name="el_grad_vti", nz=320, nx=960, nabc=40, dt=4e-4, f0=10.0, shots=48, nt=240, mode="grad",
             source="vf", vti=True),
        # sixth order, no free surface, odd sizes
        dict(el, name="el_grad_order6", nz=151, nx=333, fs=False, shots=8, nt=400, mode="grad", order=6),
        # the taper boundary (unsplit scheme)
        dict(el, name="el_grad_taper", nz=120, nx=301, shots=6, nt=400, mode="grad", abc="gerjan"),
        # the driver's misfit and its adjoint source on their own: records of a mid-sized survey
        dict(name="misfit_norm", wave="misfit", shots=24, nt=2000, rec=601, misfit="norm"),
    ]


# ---------------------------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------------------------
def _padded(case):
    a = case["nabc"]
    if case["wave"] == "acoustic":
        return case["nz"] + 2 * a, case["nx"] + 2 * a
    nn = case["order"] // 2
    return case["nz"] + (a if case["fs"] else 2 * a) + nn, case["nx"] + 2 * a


def _cost(case):
    """Relative cost: point steps, an elastic one about six acoustic ones, a modelling run about a
    quarter of a gradient."""
    if case["wave"] == "misfit":
        return 0.1 * case["shots"] * case["nt"] * case["rec"]
    Z, X = _padded(case)
    w = (1.0 if case["wave"] == "acoustic" else 6.5) * (1.0 if case["mode"] == "grad" else 0.25)
    return w * case["shots"] * case["nt"] * Z * X


def draw(rng):
    """One more case of the listed ranges: grids of 80 x 120 to 384 x 1152, 1 to 64 shots, 240 to
    1500 steps, any option, no dearer than half the largest listed case."""
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(["acoustic"] * 6 + ["elastic"] * 5 + ["misfit"])
    if kind == "misfit":
        return dict(wave="misfit", shots=log(1, 64), nt=log(500, 3000), rec=log(50, 700), misfit=rng.choice(["norm", "l2sq"]))
    limit = 3e10
    while True:
        c = dict(wave=kind, nz=log(80, 384), nx=log(120, 1152), shots=log(1, 64), nt=log(240, 1500),
                 nabc=rng.choice([20, 25, 30, 40]), fs=rng.random() < 0.5, mode=rng.choice(["model", "grad", "grad"]))
        if kind == "acoustic":
            c.update(dx=10.0, dt=1e-3, f0=10.0)
            if c["mode"] == "grad":
                c.update(misfit="l2sq", par=rng.choice(["vp", "vp", "vp+rho"]), comp=rng.choice(["p", "p", "puw"]))
        else:
            c.update(dx=5.0, dt=5e-4, f0=12.0, order=rng.choice([4, 4, 4, 6]),
                     abc=rng.choice(["PML", "PML", "PML", "gerjan"]), source=rng.choice(["mt", "vf"]),
                     vti=rng.random() < 0.4)
        if _cost(c) <= limit:
            return c


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
def _smooth_noise(g, nz, nx, scale):
    """Zero-mean smooth noise of unit standard deviation, correlated over about `scale` cells."""
    a = torch.randn(1, 1, max(3, nz // scale + 2), max(3, nx // scale + 2), generator=g)
    a = F.interpolate(a, size=(nz, nx), mode="bicubic", align_corners=True)[0, 0]
    return ((a - a.mean()) / a.std()).numpy()


def _model(case, seed):
    """vp, vs, rho, eps, delta (nz, nx) float32."""
    g = torch.Generator().manual_seed(int(seed))
    nz, nx = case["nz"], case["nx"]
    z = np.linspace(0.0, 1.0, nz)[:, None] + 0.02 * _smooth_noise(g, nz, nx, 60)
    layers = np.floor(z * 6.0) / 6.0
    vp = 1700.0 + 2200.0 * (0.5 * z + 0.5 * layers) + 120.0 * _smooth_noise(g, nz, nx, 20)
    vp = np.clip(vp, 1500.0, 4500.0)
    vs = vp / 1.73 * (1.0 + 0.03 * np.clip(_smooth_noise(g, nz, nx, 30), -1.5, 1.5))
    rho = 310.0 * vp ** 0.25 * (1.0 + 0.02 * np.clip(_smooth_noise(g, nz, nx, 30), -2, 2))
    eps = 0.1 + 0.05 * np.clip(_smooth_noise(g, nz, nx, 40), -2, 2)
    delta = 0.04 + 0.03 * np.clip(_smooth_noise(g, nz, nx, 40), -2, 2)
    return {k: v.astype(np.float32) for k, v in dict(vp=vp, vs=vs, rho=rho, eps=eps, delta=delta).items()}


def _ricker(case):
    t = np.arange(case["nt"]) * case["dt"]
    a = (math.pi * case["f0"] * (t - 1.2 / case["f0"])) ** 2
    return ((1 - 2 * a) * np.exp(-a)).astype(np.float32)


def _sources(case):
    nx, n = case["nx"], case["shots"]
    sx = np.linspace(6, nx - 7, n).astype(int) if n > 1 else np.array([nx // 3])
    return sx, np.full(n, 3)


def _arrivals(shots, nt, rec, spacing, dt, f0, src, seed, device):
    """(shots, nt, rec) float32 records: three hyperbolic arrivals and weak noise."""
    g = torch.Generator(device=device).manual_seed(int(seed) + 77)
    t = torch.arange(nt, device=device) * dt
    off = (torch.arange(rec, device=device)[None, :] - torch.as_tensor(src, device=device)[:, None]).abs() * spacing
    out = 1e-3 * torch.randn((shots, nt, rec), generator=g, device=device)
    r = np.random.default_rng(int(seed) + 78)
    for k in range(3):
        v, t0 = float(r.uniform(1600, 3000)), float(r.uniform(0.0, 0.3)) * k * nt * dt
        tt = torch.sqrt(t0 ** 2 + (off / v) ** 2) + 1.2 / f0
        a = (math.pi * f0 * (t[None, :, None] - tt[:, None, :])) ** 2
        out += float(r.uniform(0.4, 1.0)) * (1 - 2 * a) * torch.exp(-a) / torch.sqrt(1.0 + off / (20 * spacing))[:, None, :]
    return out


def _components(case):
    if case["wave"] == "elastic":
        return ["vx", "vz"]
    return list(case["comp"])


def _observed(case, seed, device):
    sx, _ = _sources(case)
    scale = (1e-3 if case["wave"] == "acoustic" else 1e-1 if case["source"] == "vf" else 1e-7)
    obs = {}
    for i, k in enumerate(_components(case)):
        o = _arrivals(case["shots"], case["nt"], case["nx"], case["dx"], case["dt"], case["f0"], sx, seed + 1000 * i, device)
        # particle velocities are smaller than pressures by the impedance
        obs[k] = o * (scale * (2e-7 if case["wave"] == "acoustic" and k != "p" else 1.0))
    if case["misfit_kind"] == "norm":
        obs = {k: o / o.abs().amax(1, keepdim=True) for k, o in obs.items()}
    return obs


def _misfit_kind(case):
    return case.get("misfit", "l2sq")


def prepare(case, seed):
    from adfwi_amd.fwi import Misfit_waveform_L2_squared, NormalizedWaveformL2
    kind = _misfit_kind(case)
    if case["wave"] == "misfit":
        syn, obs = _records(case, seed, DEV)
        fn = (NormalizedWaveformL2 if kind == "norm" else Misfit_waveform_L2_squared)(1e-3)
        return {"case": case, "syn": syn.requires_grad_(True), "obs": obs, "misfit": fn}
    from adfwi_amd.model import AcousticModel, AnisotropicElasticModel, IsotropicElasticModel
    from adfwi_amd.propagator import AcousticPropagator, ElasticPropagator
    from adfwi_amd.survey import Receiver, Source, Survey
    m = _model(case, seed)
    grad = case["mode"] == "grad"
    nz, nx = case["nz"], case["nx"]
    sx, sz = _sources(case)
    src = Source(case["nt"], case["dt"], case["f0"])
    src.add_sources(sx, sz, _ricker(case), "mt" if case["wave"] == "acoustic" else case["source"])
    rcv = Receiver(case["nt"], case["dt"])
    rcv.add_receivers(np.arange(nx), np.full(nx, 2), "pr" if case["wave"] == "acoustic" else "vz")
    survey = Survey(src, rcv)
    if case["wave"] == "acoustic":
        model = AcousticModel(0, 0, nx, nz, case["dx"], case["dx"], vp=m["vp"], rho=m["rho"], vp_grad=grad,
                              rho_grad=grad and case["par"] == "vp+rho", nabc=case["nabc"], free_surface=case["fs"],
                              device=DEV)
        prop = AcousticPropagator(model, survey, device=DEV)
        pars = ["vp"] + (["rho"] if grad and case["par"] == "vp+rho" else [])
    else:
        common = dict(free_surface=case["fs"], nabc=case["nabc"], auto_update_rho=False, abc_type=case["abc"],
                      device=DEV, vp_grad=grad, vs_grad=grad, rho_grad=grad)
        if case["vti"]:
            model = AnisotropicElasticModel(0, 0, nx, nz, case["dx"], case["dx"], vp=m["vp"], vs=m["vs"], rho=m["rho"],
                                            eps=m["eps"], gamma=np.zeros_like(m["vp"]), delta=m["delta"],
                                            eps_grad=grad, delta_grad=grad, **common)
            pars = ["vp", "vs", "rho", "eps", "delta"]
        else:
            model = IsotropicElasticModel(0, 0, nx, nz, case["dx"], case["dx"], vp=m["vp"], vs=m["vs"], rho=m["rho"],
                                          **common)
            pars = ["vp", "vs", "rho"]
        prop = ElasticPropagator(model, survey, device=DEV)
    state = {"case": case, "model": model, "prop": prop, "pars": pars}
    if grad:
        state["obs"] = _observed(dict(case, misfit_kind=kind), seed, DEV)
        state["misfit"] = (NormalizedWaveformL2 if kind == "norm" else Misfit_waveform_L2_squared)(case["dt"])
    return state


def _records(case, seed, device):
    """Synthetic and (normalised) observed records of a misfit case."""
    S, nt, R = case["shots"], case["nt"], case["rec"]
    src = np.linspace(0, R - 1, S).astype(int)
    syn = _arrivals(S, nt, R, 12.5, 1e-3, 10.0, src, seed, device)
    obs = _arrivals(S, nt, R, 12.5, 1e-3, 10.0, src, seed + 5000, device)
    if _misfit_kind(case) == "norm":
        obs = obs / obs.abs().amax(1, keepdim=True)
    return syn, obs


def run(state):
    case = state["case"]
    if case["wave"] == "misfit":
        syn = state["syn"]
        syn.grad = None
        loss = state["misfit"].forward(syn, state["obs"])
        loss.backward()
        return {"loss": loss.detach(), "grad": syn.grad}
    model, prop = state["model"], state["prop"]
    kw = {"fd_order": case["order"]} if case["wave"] == "elastic" else {}
    if case["mode"] == "model":
        with torch.no_grad():
            return prop.forward(**kw)
    for par in state["pars"]:
        getattr(model, par).grad = None
    rec = prop.forward(**kw)
    loss = sum(state["misfit"].forward(rec[k], state["obs"][k]) for k in state["obs"])
    loss.backward()
    out = {k: v.detach() for k, v in rec.items()}
    out["loss"] = loss.detach()
    for par in state["pars"]:
        out["grad_" + par] = getattr(model, par).grad
    return out


def work(case):
    """Bytes: models, observed data, records, maps and gradients, once each.  Flops: the update
    formulas' own operations per point and step (acoustic forward 28 + 4 for the energy maps,
    adjoint with imaging 45; elastic forward 85, adjoint with imaging 190; half of that for the
    unsplit scheme), without any recomputation."""
    if case["wave"] == "misfit":
        n = case["shots"] * case["nt"] * case["rec"]
        return {"bytes": 12.0 * n, "flops": 12.0 * n}
    Z, X = _padded(case)
    pts = float(case["shots"]) * case["nt"] * Z * X
    grad = case["mode"] == "grad"
    ac = case["wave"] == "acoustic"
    ncomp = 3 if ac else 5
    rec = 4.0 * case["shots"] * case["nt"] * case["nx"]
    maps = 4.0 * case["nz"] * case["nx"]
    npar = 2 if ac else (5 if case["vti"] else 3)
    nbytes = rec * ncomp + maps * (npar + ncomp)
    flops = pts * (32 if ac else 85 if case["abc"] == "PML" else 60)
    if grad:
        nbytes += 2 * rec * len(_components(case)) + maps * npar
        flops += pts * (45 if ac else 190 if case["abc"] == "PML" else 130)
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------------------------
# the same in 64 bits, from the update formulas, in plain torch
# ---------------------------------------------------------------------------------------------
def _edge_pad(a, left, right, top, bottom):
    return F.pad(a[None, None], (left, right, top, bottom), mode="replicate")[0, 0]


def _shift(a, dz, dx):
    """a[..., i + dz, j + dx] (wraps at the borders, where every use is masked)."""
    return torch.roll(a, (-dz, -dx), (-2, -1))


def _embed(a, Z, X):
    return F.pad(a, (0, X - a.shape[1], 0, Z - a.shape[0]))


def _window(Z, X, r0, r1, c0, c1, dev):
    m = torch.zeros((Z, X), dtype=torch.float64, device=dev)
    m[r0:r1, c0:c1] = 1.0
    return m


def _march(step, state, nt, consts, grad):
    """All steps; each chunk recomputed in the backward.  Returns per-step outputs stacked over time."""
    k = max(1, int(math.sqrt(nt)))
    outs = []

    def chunk(t0, n, *a):
        st, cs = list(a[:len(state)]), a[len(state):]
        got = []
        for t in range(t0, t0 + n):
            st, o = step(t, st, cs)
            got.append(o)
        return (*st, *[torch.stack(x) for x in zip(*got)])

    st = list(state)
    for t0 in range(0, nt, k):
        n = min(k, nt - t0)
        r = checkpoint(chunk, t0, n, *st, *consts, use_reentrant=False) if grad else chunk(t0, n, *st, *consts)
        st, o = list(r[:len(state)]), r[len(state):]
        outs.append(o)
    return st, [torch.cat(x) for x in zip(*outs)]


def _exact_acoustic(case, m, dev, pars):
    d = torch.float64
    nz, nx, a, dx, dt, nt = case["nz"], case["nx"], case["nabc"], case["dx"], case["dt"], case["nt"]
    Z, X = _padded(case)
    fs = a if case["fs"] else 1
    vp = torch.tensor(m["vp"], dtype=d, device=dev).requires_grad_("vp" in pars)
    # the model's density is Gardner's of its vp, a parameter of its own
    rho = (310.0 * vp.detach() ** 0.25).requires_grad_("rho" in pars)
    depth = torch.arange(a, dtype=d, device=dev) * dx / ((a - 1) * dx)
    prof = 3.0 * float(m["vp"].max()) * math.log(1e6) / (2.0 * (a - 1) * dx) * depth ** 2
    rows, cols = torch.arange(Z, device=dev)[:, None], torch.arange(X, device=dev)[None, :]
    kz = torch.maximum(a - 1 - rows, rows - (Z - a))          # depth index into the z strips
    kx = torch.maximum(a - 1 - cols, cols - (X - a))
    damp = torch.where((kx >= 0).expand(Z, X), prof[kx.clamp(0, a - 1)].expand(Z, X), torch.zeros((), dtype=d, device=dev))
    # a z strip of depth kz covers the columns up to that depth of the x strips
    inz = (kz >= 0) & (cols >= a - kz) & (cols < X - a + kz)
    damp = torch.where(inz, prof[kz.clamp(0, a - 1)].expand(Z, X), damp)
    c, den = _edge_pad(vp, a, a, a, a), _edge_pad(rho, a, a, a, a)
    a1, a2 = den * c * c * dt / dx, dt / (den * dx)
    k1 = damp * dt
    k2 = torch.zeros_like(damp)
    k2[:, 1:X - 2] = 0.5 * (damp[:, 1:X - 2] + damp[:, 2:X - 1]) * dt
    k3 = torch.zeros_like(damp)
    k3[fs:Z - 2] = 0.5 * (damp[fs:Z - 2] + damp[fs + 1:Z - 1]) * dt
    mp = _window(Z, X, fs + 1, Z - 2, 2, X - 2, dev)
    mu = _window(Z, X, fs, Z - 1, 1, X - 2, dev)
    mw = _window(Z, X, fs, Z - 2, 1, X - 1, dev)
    top = _window(Z, X, fs - 1, fs, 0, X, dev) if case["fs"] else None
    sx, sz = (torch.as_tensor(v, device=dev) + a for v in _sources(case))
    S = case["shots"]
    at = torch.zeros((S, Z, X), dtype=d, device=dev)
    at[torch.arange(S, device=dev), sz, sx] = 1.0
    wav = torch.tensor(_ricker(case), dtype=d, device=dev) * dt
    rx, rz = torch.arange(nx, device=dev) + a, torch.full((nx,), 2 + a, device=dev)
    C1, C2 = 9.0 / 8.0, -1.0 / 24.0
    crop = (slice(None), slice(a, a + nz), slice(a, a + nx))

    def step(t, st, cs):
        p, u, w = st
        b1, b2, b3, a1m, a2u, a2w = cs
        dd = (C1 * (u - _shift(u, 0, -1) + w - _shift(w, -1, 0))
              + C2 * (_shift(u, 0, 1) - _shift(u, 0, -2) + _shift(w, 1, 0) - _shift(w, -2, 0)))
        p = b1 * p - a1m * dd + at * wav[t]
        if top is not None:
            p = p * (1.0 - top) - _shift(p, 2, 0) * top
        u = b2 * u - a2u * (C1 * (_shift(p, 0, 1) - p) + C2 * (_shift(p, 0, 2) - _shift(p, 0, -1)))
        w = b3 * w - a2w * (C1 * (_shift(p, 1, 0) - p) + C2 * (_shift(p, 2, 0) - _shift(p, -1, 0)))
        if top is not None:
            w = w * (1.0 - top) + _shift(w, 1, 0) * top
        en = [(v.detach()[crop] ** 2).sum(0) for v in (p, u, w)]
        return [p, u, w], [p[:, rz, rx], u[:, rz, rx], w[:, rz, rx], *en]

    zero = torch.zeros((S, Z, X), dtype=d, device=dev)
    consts = (1.0 - k1 * mp, 1.0 - k2 * mu, 1.0 - k3 * mw, a1 * mp, a2 * mu, a2 * mw)
    _, o = _march(step, [zero, zero, zero], nt, consts, bool(pars))
    rec = {k: o[i].transpose(0, 1) for i, k in enumerate("puw")}
    ep, eu, ew = o[3].sum(0), o[4].sum(0), o[5][-1]
    maps = {"forward_wavefield_p": ep, "forward_wavefield_u": ep + eu, "forward_wavefield_w": ep + eu + ew}
    return rec, maps, {"vp": vp, "rho": rho}


def _fd_coefs(n):
    """The staggered difference's coefficients of half-order n; at most three of them are used."""
    A = np.array([[(2 * j + 1) ** (2 * i + 1) for j in range(n)] for i in range(n)], dtype=np.float64)
    return list(np.linalg.solve(A, np.eye(n)[0]))[:3]


def _exact_elastic(case, m, dev, pars):
    d = torch.float64
    nz, nx, a, dx, dt, nt, fs = (case[k] for k in ("nz", "nx", "nabc", "dx", "dt", "nt", "fs"))
    nn = case["order"] // 2
    Z, X = _padded(case)
    S = case["shots"]
    par = {k: torch.tensor(m[k], dtype=d, device=dev).requires_grad_(k in pars) for k in ("vp", "vs", "rho", "eps", "delta")}
    vp, vs, rho = par["vp"], par["vs"], par["rho"]
    eps, delta = (par["eps"], par["delta"]) if case["vti"] else (torch.zeros_like(vp), torch.zeros_like(vp))
    c33, c44 = vp ** 2 * rho, vs ** 2 * rho
    c11 = c33 * (1 + 2 * eps)
    c13 = torch.sqrt(2 * c33 * (c33 - c44) * delta + (c33 - c44) ** 2) - c44
    b = 1.0 / rho
    bx, bz = 0.5 * (b[:, :-1] + b[:, 1:]), 0.5 * (b[:-1] + b[1:])
    c55 = 0.2 * (c44[1:-1, 1:-1] + 2 * c44[2:, 1:-1] + c44[1:-1, 2:] + c44[2:, 2:])
    top = nn if fs else a + nn
    win = _window(Z, X, nn, Z - nn, nn, X - nn, dev)
    pad = lambda v: _embed(_edge_pad(v, a, a, top, a), Z, X) * win
    C11, C13, C33, C55, BX, BZ = (pad(v) for v in (c11, c13, c33, c55, bx, bz))
    fd = _fd_coefs(nn)
    dif = lambda v, ax, fwd: sum(cf * (_shift(v, *(((k + fwd), 0) if ax == 0 else (0, k + fwd)))
                                       - _shift(v, *((fwd - 1 - k, 0) if ax == 0 else (0, fwd - 1 - k))))
                                 for k, cf in enumerate(fd))
    dxf, dxb = (lambda v: dif(v, 1, 1)), (lambda v: dif(v, 1, 0))
    dzf, dzb = (lambda v: dif(v, 0, 1)), (lambda v: dif(v, 0, 0))
    h = nn + 1
    row = lambda r, w0=0, w1=X: _window(Z, X, r, r + 1, w0, w1, dev)
    r0, r1, r2 = row(h - 3), row(h - 2), row(h - 1)
    j0, j1 = row(h - 3, nn, X - nn), row(h - 2, nn, X - nn)

    def fs_stress(tzz, txz):
        tzz = tzz * (1 - r2)
        tzz = tzz * (1 - r1) - _shift(tzz, 2, 0) * r1
        new = txz * (1 - r1) - _shift(txz, 1, 0) * r1
        return tzz, new * (1 - r0) - _shift(txz, 3, 0) * r0

    def fs_vel(vx, vz):
        vz = vz * (1 - j1) + _shift(vz, 1, 0) * j1
        new = (_shift(vz, 0, 1) - vz) + (_shift(vz, 1, 1) - _shift(vz, 1, 0)) + _shift(vx, 2, 0)
        vx = vx * (1 - j1) + new * j1
        return vx, vz * (1 - j0) + _shift(vz, 1, 0) * j0

    sx, sz = _sources(case)
    sx, sz = torch.as_tensor(sx, device=dev) + a, torch.as_tensor(sz, device=dev) + top
    at = torch.zeros((S, Z, X), dtype=d, device=dev)
    at[torch.arange(S, device=dev), sz, sx] = 1.0
    wav = torch.tensor(_ricker(case), dtype=d, device=dev)
    mt, vf = (1.0, 0.0) if case["source"] == "mt" else (0.0, 1.0)
    rx, rz = torch.arange(nx, device=dev) + a, torch.full((nx,), 2 + top, device=dev)
    crop = (slice(None), slice(top, top + nz), slice(a, a + nx))
    zero = torch.zeros((S, Z, X), dtype=d, device=dev)

    def results(txx, tzz, txz, vx, vz):
        f = (txx, tzz, txz, vx, vz)
        return [v[:, rz, rx] for v in f] + [(v.detach()[crop] ** 2).sum(0) for v in f]

    if case["abc"] == "PML":
        k = torch.arange(1, a + 1, dtype=d, device=dev)
        prof = (a - k + 1) ** 2 * (math.log(1e6) * 3 * float(m["vp"].max()) / (2 * a ** 3)) / dx
        px, pz = torch.zeros(X, dtype=d, device=dev), torch.zeros(Z, dtype=d, device=dev)
        px[:a], px[X - a:] = prof, prof.flip(0)
        if not fs:
            pz[nn:nn + a] = prof
            pz[:nn] = prof[0]                    # the rows above repeat the profile's first
        pz[Z - a:] = prof.flip(0)
        xn, xd = 1 - 0.5 * dt * px, 1 + 0.5 * dt * px
        zn, zd = (1 - 0.5 * dt * pz)[:, None], (1 + 0.5 * dt * pz)[:, None]
        keep = lambda new, old: new * win + old * (1 - win)

        def step(t, st, cs):
            c11_, c13_, c33_, c55_, bx_, bz_ = cs
            (xxx, xxz, zzx, zzz, xzx, xzz, vxx, vxz, vzx, vzz) = st
            vx, vz = vxx + vxz, vzx + vzz
            if fs:
                vx, vz = fs_vel(vx, vz)
            s = at * (-0.5 * mt * wav[t])
            q = dt / dx
            xxx = (xn * xxx + q * c11_ * dxb(vx)) / xd * win + s
            xxz = (zn * xxz + q * c13_ * dzb(vz)) / zd * win + s
            zzx = (xn * zzx + q * c13_ * dxb(vx)) / xd * win + s
            zzz = (zn * zzz + q * c33_ * dzb(vz)) / zd * win + s
            xzx = (xn * xzx + q * c55_ * dxf(vz)) / xd * win
            xzz = (zn * xzz + q * c55_ * dzf(vx)) / zd * win
            txx, tzz, txz = xxx + xxz, zzx + zzz, xzx + xzz
            if fs:
                tzz, txz = fs_stress(tzz, txz)
            f = at * (0.5 * vf * wav[t])
            vxx = (xn * vxx + q * bx_ * dxf(txx)) / xd * win
            vxz = (zn * vxz + q * bx_ * dzb(txz)) / zd * win
            vzx = (xn * vzx + q * bz_ * dxb(txz)) / xd * win + f
            vzz = (zn * vzz + q * bz_ * dzf(tzz)) / zd * win + f
            vx, vz = vxx + vxz, vzx + vzz
            if fs:
                vx, vz = fs_vel(vx, vz)
            return [xxx, xxz, zzx, zzz, xzx, xzz, vxx, vxz, vzx, vzz], results(txx, tzz, txz, vx, vz)
        state = [zero] * 10
    else:
        wt = np.exp(-(0.0053 * (a - np.arange(1, a + 1))) ** 2)
        rows, cols = np.arange(Z - nn)[:, None], np.arange(X)[None, :]
        depth = np.minimum(np.minimum(cols, X - 1 - cols), Z - nn - 1 - rows)
        if not fs:
            depth = np.minimum(depth, rows)
        dm = np.where(depth < a, wt[np.minimum(depth, a - 1)], 1.0)
        taper = torch.tensor(np.concatenate([np.repeat(dm[:1], nn, 0), dm], 0), dtype=d, device=dev)

        def step(t, st, cs):
            c11_, c13_, c33_, c55_, bx_, bz_ = cs
            txx, tzz, txz, vx, vz = st
            s = at * (-mt / 3.0 * wav[t])
            q = dt / dx
            txx = txx + q * (c11_ * dxb(vx) + c13_ * dzb(vz)) + s
            tzz = tzz + q * (c13_ * dxb(vx) + c33_ * dzb(vz)) + s
            txz = txz + q * (c55_ * dxf(vz) + c55_ * dzf(vx))
            if fs:
                tzz, txz = fs_stress(tzz, txz)
            vx = vx + q * bx_ * (dxf(txx) + dzb(txz))
            vz = vz + q * bz_ * (dxb(txz) + dzf(tzz)) + at * (vf * wav[t])
            if fs:
                vx, vz = fs_vel(vx, vz)
            vx, vz = vx * taper, vz * taper
            return [txx, tzz, txz, vx, vz], results(txx, tzz, txz, vx, vz)
        state = [zero] * 5
    _, o = _march(step, state, nt, (C11, C13, C33, C55, BX, BZ), bool(pars))
    names = ("txx", "tzz", "txz", "vx", "vz")
    rec = {k: o[i].transpose(0, 1) for i, k in enumerate(names)}
    maps = {"forward_wavefield_" + k: o[5 + i][-1] for i, k in enumerate(names)}
    return rec, maps, par


def _exact_misfit(kind, syn, obs, dt):
    if kind == "norm":
        syn = syn / syn.abs().amax(1, keepdim=True)
        return torch.sqrt(((obs - syn) ** 2 * dt).sum(1)).sum()
    return 0.5 * dt * ((obs - syn) ** 2).sum()


def exact(case, seed):
    """run()'s outputs in 64 bits; None for cases whose 64-bit autograd takes too long."""
    dev = DEV if torch.cuda.is_available() else "cpu"
    kind = _misfit_kind(case)
    if case["wave"] == "misfit":
        syn, obs = (x.to(torch.float64) for x in _records(case, seed, dev))
        syn.requires_grad_(True)
        loss = _exact_misfit(kind, syn, obs, 1e-3)
        loss.backward()
        return {"loss": loss.detach(), "grad": syn.grad}
    grad = case["mode"] == "grad"
    if _cost(case) > (4.0e9 if grad else 2.0e9):
        return None
    m = _model(case, seed)
    if not grad:
        pars = []
    elif case["wave"] == "acoustic":
        pars = ["vp"] + (["rho"] if case["par"] == "vp+rho" else [])
    else:
        pars = ["vp", "vs", "rho"] + (["eps", "delta"] if case["vti"] else [])
    with torch.set_grad_enabled(grad):
        rec, maps, leaf = (_exact_acoustic if case["wave"] == "acoustic" else _exact_elastic)(case, m, dev, pars)
        out = {k: v.detach() for k, v in (rec | maps).items()}
        if grad:
            obs = _observed(dict(case, misfit_kind=kind), seed, dev)
            loss = sum(_exact_misfit(kind, rec[k], obs[k].to(torch.float64), case["dt"]) for k in obs)
            loss.backward()
            out["loss"] = loss.detach()
            for par in pars:
                out["grad_" + par] = leaf[par].grad
    return out
