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
