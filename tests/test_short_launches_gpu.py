"""Runs whose launches are cut to one and two steps (checkpoints that close together, ends of calls)
on grids of more than one and more than eight rounds of tile workgroups, where those go to the strip
kernels, against the one-step kernels: records, final state and checkpoints bit for bit, gradients to
rounding.

Tolerance: N = 16 steps * 600 shots terms per point, each addition rounding to 2^-24: sqrt(9600) *
2^-24 = 5.8e-6; twice that leaves room for cancellation.
"""
import numpy as np
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("k", [1, 2, 5, 6])
@pytest.mark.parametrize("Z,X,S,fs", [(41, 105, 70, 0), (41, 105, 600, 5), (48, 80, 300, 0)])
def test_short_launches_equal_one_step_kernels(monkeypatch, Z, X, S, fs, k):
    from adfwi_amd.propagator import acoustic_kernels as ak
    rng = np.random.default_rng(Z * 1000 + X)
    lo, nt = max(fs, 1), 16
    src_z, src_x = rng.integers(lo, Z - 1, S), rng.integers(1, X - 1, S)
    rx = np.arange(0, X - 1, 2)
    gen = torch.Generator().manual_seed(Z + X)
    field = lambda a, b: (a + (b - a) * torch.rand((Z, X), generator=gen)).to(DEV)
    a1, a2, omk = field(0.1, 0.3), field(0.1, 0.3), [field(0.9, 1.0) for _ in range(3)]
    src = torch.randn((S, nt), generator=gen).to(DEV)
    adj = torch.randn((S, nt, len(rx)), generator=gen).to(DEV)
    out = []
    for fuse in ("0", "1"):
        monkeypatch.setenv("ADFWI_FUSE_STEPS", fuse)
        g = ak.AcousticGeometry(Z, X, nt, bool(fs), fs if fs else 1, src_z, src_x, np.full(len(rx), lo + 1), rx, DEV)
        coef = g.pack_coef(omk[0], a1, omk[1], a2, omk[2])
        res = ak.run_forward(g, coef, src, ckpt_every=k, energy_u_from=5)
        ck = None if res["ckpt"] is None else res["ckpt"].cpu().numpy()
        grads = ak.run_backward(g, coef, src, res["ckpt"], k, (adj, None, None), True, False, True)
        out.append(([r.cpu().numpy() for r in res["rec"]], ck, res["energy"].cpu().numpy(), grads[0].cpu().numpy(),
                    grads[2].cpu().numpy()))
    (r0, c0, e0, g0, w0), (r1, c1, e1, g1, w1) = out
    for i in range(3):
        same = np.array_equal(r0[i], r1[i])
        assert same, ("record", i)
    same = np.array_equal(c0, c1), np.array_equal(w0, w1)
    assert same == (True, True)
    for a, b in ((e1[0], e0[0]), (e1[1], e0[1]), (g1, g0)):
        err = rel_l2(a, b)
        assert np.abs(b).max() > 0 and err <= 1.2e-5, err


@pytest.mark.parametrize("resident", [0, 4])
@pytest.mark.parametrize("Z,X,S", [(60, 60, 65), (64, 60, 80)])     # 260 and 320 tiles of 52 x 52 points
def test_elastic_segments_of_one_step_keep_splits(Z, X, S, resident):
    """At 4th order and more than one round of tiles, checkpoints after every step take the step kernels'
    adjoint and their traces: gradients as of longer segments of totals, to rounding (13 steps of at most
    80 shots: sqrt(1040) * 2^-24 = 1.9e-6; 5e-6 leaves room for cancellation), and the wavelet's bits."""
    from adfwi_amd.propagator import elastic_adjoint as ea
    from adfwi_amd.propagator import elastic_kernels as ek
    rng, nt = np.random.default_rng(Z), 13
    gen = torch.Generator().manual_seed(S)
    rand = lambda a, b, *shape: a + (b - a) * torch.rand(shape, generator=gen)
    rx = np.arange(2, X - 2, 3)
    g = ek.ElasticGeometry(Z, X, nt, True, rng.integers(2, Z - 2, S), rng.integers(2, X - 2, S), rand(-1, 1, S, 3),
                           np.full(len(rx), 3), rx, DEV, resident_traces=resident)
    assert g.totals and g.trace_totals(2) and not g.trace_totals(1)
    scalars = (1e-2, 2e-2, 2.5e-2, 0.5, 0.4, 1.125, -1.0 / 24)
    px, pz = (t.to(DEV) for t in ek.pml_factors(rand(0, 20, 1, X).expand(Z, X), rand(0, 20, Z, 1).expand(Z, X),
                                                scalars[0], g.pitch))
    coef = g.pack_coef([rand(a, b, Z, X).to(DEV) for a, b in ((5, 9), (1, 3), (5, 9), (1, 3), (.3, .6), (.3, .6))]
                       + [None, None])
    src = rand(-1, 1, S, nt).to(DEV)
    adj = [rand(-1, 1, S, nt, len(rx)).to(DEV) for _ in range(5)]
    out = []
    for k in (1, 5):
        res = ek.run_forward(g, coef, px, pz, src, scalars, ckpt_every=k, resident=min(resident, -(-nt // k)))
        assert res["totals"] == (k > 1)
        out.append((res["rec"], ea.run_backward(g, coef, src, px, pz, scalars, res["ckpt"], k, adj,
                                                [True] * 6 + [False] * 2 + [True], traces=res["traces"])))
    (ra, (ga, wa)), (rb, (gb, wb)) = out
    for i in range(5):
        assert torch.equal(ra[i], rb[i]), ("record", i)
    for i in range(6):
        err = rel_l2(ga[i].cpu().numpy(), gb[i].cpu().numpy())
        assert gb[i].abs().max() > 0 and err <= 5e-6, ("gradient", i, err)
    assert torch.equal(wa, wb)
