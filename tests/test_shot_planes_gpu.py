"""Energy and gradient planes of the acoustic kernels that a caller keeps apart: plane g holds the
shots of group g and no others, also where the launch would take more shots together for a sum
(grids of over 256 tile workgroups), and so a packed request's gradient is its own.

Tolerance: at most N = 37 steps * 2 shots (planes) or 90 steps * 15 shots (requests) terms per
point, each addition rounding to 2^-24: sqrt(1350) * 2^-24 = 2.2e-6; 5e-6 leaves room for
cancellation.  A shot in another plane changes it by a large part of its size.
"""
import copy
import ctypes

import numpy as np
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# Z, X, shots, free-surface row: groups of 2 (the last one shot) and of 3 shots where planes are
# summed, and of 2 with the rho gradient
CASES = [(41, 105, 81, 0), (41, 105, 161, 5)]


def _problem(monkeypatch, Z, X, S, fs, fuse):
    from adfwi_amd.propagator import acoustic_kernels as ak
    monkeypatch.setenv("ADFWI_FUSE_STEPS", fuse)
    rng = np.random.default_rng(Z * 1000 + X)
    lo = max(fs, 1)
    src_z, src_x = rng.integers(lo, Z - 1, S), rng.integers(1, X - 1, S)
    rx = np.arange(0, X - 1, 2)
    nt = 37
    g = ak.AcousticGeometry(Z, X, nt, bool(fs), fs if fs else 1, src_z, src_x, np.full(len(rx), lo + 1), rx, DEV)
    gen = torch.Generator().manual_seed(Z + X)
    field = lambda a, b: (a + (b - a) * torch.rand((Z, X), generator=gen)).to(DEV)
    a1, a2 = field(0.1, 0.3), field(0.1, 0.3)
    coef = g.pack_coef(field(0.9, 1.0), a1, field(0.9, 1.0), a2, field(0.9, 1.0))
    return ak, g, coef, torch.randn((S, nt), generator=gen).to(DEV), torch.randn((S, nt, len(rx)), generator=gen).to(DEV)


@pytest.mark.parametrize("rho", [False, True])
@pytest.mark.parametrize("Z,X,S,fs", CASES)
def test_gradient_planes_hold_their_own_shots(monkeypatch, Z, X, S, fs, rho):
    out = []
    for fuse in ("0", "1"):
        ak, g, coef, src, adj = _problem(monkeypatch, Z, X, S, fs, fuse)
        res = ak.run_forward(g, coef, src, ckpt_every=11, resident=1, need_a1=True, need_a2=rho)
        planes = ak.run_backward(g, coef, src, res["ckpt"], 11, (adj, None, None), True, rho, False,
                                 group_planes=True, images=res["images"])
        assert planes[0].shape[0] == -(-S // g.gradient_group)
        out.append([p.cpu().numpy() for p in planes[:2] if p is not None])
    for name, a, b in zip(("a1", "a2"), out[1], out[0]):
        for i, (x, y) in enumerate(zip(a, b)):
            assert np.abs(y).max() > 0 and rel_l2(x, y) <= 5e-6, (name, i, rel_l2(x, y))


@pytest.mark.parametrize("Z,X,S,fs", CASES)
def test_energy_planes_hold_their_own_shots(monkeypatch, Z, X, S, fs):
    from adfwi_amd import _native as nat
    out = []
    for fuse in ("0", "1"):
        ak, g, coef, src, _ = _problem(monkeypatch, Z, X, S, fs, fuse)
        work = g.state(2)
        energy = torch.zeros((int(g.layout.ngroups), 2, Z, g.pitch), device=DEV)
        d, a = g.desc(coef, src), nat.AcousticFwdArgs()
        a.state_in = work[0].data_ptr()
        a.work[0], a.work[1] = work[0].data_ptr(), work[1].data_ptr()
        a.t0, a.nsteps, a.energy_u_from, a.energy = 0, g.nt, 5, energy.data_ptr()
        a.rcv_map, a.fuse_steps = g.rcv_map.data_ptr() if g.rcv_map is not None else None, g.fuse_steps
        nat.check(nat.load().adfwi_acoustic_forward(ctypes.byref(d), ctypes.byref(a), nat.stream_handle(energy.device)),
                  "adfwi_acoustic_forward")
        out.append(energy.cpu().numpy())
    for i in range(out[0].shape[0]):
        for q in range(2):
            x, y = out[1][i, q], out[0][i, q]
            assert np.abs(y).max() > 0 and rel_l2(x, y) <= 5e-6, (i, q, rel_l2(x, y))


def test_packed_gradients_of_many_shots_equal_their_results_alone():
    """One shared model, members of 8, 6, 3 and 15 shots: over 256 tile workgroups together."""
    from adfwi_amd.serving import Request, ServingLoop, run_alone
    reqs = [Request(i, "acoustic", "gradient", 128, 288, 90, ns, 5000 + i, 0.0, 20, keep=True, model=505)
            for i, ns in enumerate((8, 6, 3, 15))]
    rep = ServingLoop(DEV, max_slots=1, graph_steps=0).run(copy.deepcopy(reqs), realtime=False)
    assert all(o.error is None for o in rep.outcomes), [o.error for o in rep.outcomes]
    assert any(len(p) == 4 for p in rep.packs), rep.packs
    for a, b in zip(rep.outcomes, run_alone(reqs, DEV)):
        assert a.rid == b.rid and a.result.keys() == b.result.keys()
        for k in b.result:
            x, y = a.result[k].detach().cpu().numpy(), b.result[k].detach().cpu().numpy()
            assert np.abs(y).max() > 0 and rel_l2(x, y) <= 5e-6, (a.rid, k, rel_l2(x, y))
