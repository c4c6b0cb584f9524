"""The images that the acoustic forward writes for the adjoint, for every null pattern of the two image
pointers, against the one-step kernels: the pressure image at every point and the stencil image at
every point that the pressure update changes (the adjoint uses no others) are the same bits, and so
are states and records.  And the gradient of A2 alone, for which the forward and the recomputation
write the pressure image without the stencil image.

Tolerance of that gradient: N = 37 steps * 12 shots terms per point in another order, each addition
rounding to 2^-24: sqrt(444) * 2^-24 = 1.3e-6; 5e-6 leaves room for cancellation.
"""
import ctypes

import numpy as np
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# Z, X, shots, free-surface row: tiles of 40 x 64, 64 x 64 and 64 x 128 points, odd widths, the last
# tile one column short, groups of two shots
CASES = [(8, 8, 1, 0), (33, 81, 2, 0), (121, 200, 12, 0), (40, 208, 63, 6), (79, 103, 64, 0), (41, 105, 81, 5)]


def forward(monkeypatch, Z, X, S, fs, fuse, image, image_p, records):
    from adfwi_amd import _native as nat
    from adfwi_amd.propagator import acoustic_kernels as ak
    monkeypatch.setenv("ADFWI_FUSE_STEPS", fuse)
    rng = np.random.default_rng(Z * 1000 + X)
    lo = max(fs, 1)
    rx = np.arange(0, X - 1, 2)
    gen = torch.Generator().manual_seed(Z + X)
    g = ak.AcousticGeometry(Z, X, 37, bool(fs), fs if fs else 1, rng.integers(lo, Z - 1, S), rng.integers(1, X - 1, S),
                            np.full(len(rx), lo + 1), rx, DEV)
    field = lambda a, b: (a + (b - a) * torch.rand((Z, X), generator=gen)).to(DEV)
    coef = g.pack_coef(field(0.9, 1.0), field(0.1, 0.3), field(0.9, 1.0), field(0.1, 0.3), field(0.9, 1.0))
    src = torch.randn((S, g.nt), generator=gen).to(DEV)
    n, work = 11, g.state(2)                         # launches of 4, 4 and 3 steps
    img, imp = (torch.zeros((n, S, Z, g.pitch), device=DEV) if w else None for w in (image, image_p))
    rec = [torch.zeros((S, g.nt, g.R), device=DEV) for _ in range(3)] if records else []
    d, a = g.desc(coef, src), nat.AcousticFwdArgs()
    a.state_in = work[0].data_ptr()
    a.work[0], a.work[1] = work[0].data_ptr(), work[1].data_ptr()
    a.t0, a.nsteps, a.energy_u_from, a.fuse_steps = 0, n, g.nt, g.fuse_steps
    a.image, a.image_p = (None if t is None else t.data_ptr() for t in (img, imp))
    if records:
        a.rec_p, a.rec_u, a.rec_w = (r.data_ptr() for r in rec)
    a.rcv_map = None if g.rcv_map is None else g.rcv_map.data_ptr()
    nat.check(nat.load().adfwi_acoustic_forward_sum(ctypes.byref(d), ctypes.byref(a), nat.stream_handle(src.device)),
              "adfwi_acoustic_forward")
    state = work[0] if a.state_out == work[0].data_ptr() else work[1]
    if image:
        img = img[:, :, g.fs + 1:Z - 2, 2:X - 2]     # the window of the pressure update
    return [t.cpu().numpy() for t in [state] + [t for t in (img, imp) if t is not None] + rec]


@pytest.mark.parametrize("records", [False, True])
@pytest.mark.parametrize("image,image_p", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("Z,X,S,fs", CASES)
def test_images_equal_one_step_kernels(monkeypatch, Z, X, S, fs, image, image_p, records):
    one, tiles = (forward(monkeypatch, Z, X, S, fs, fuse, image, image_p, records) for fuse in ("0", "1"))
    for i, (x, y) in enumerate(zip(tiles, one)):
        err = rel_l2(x, y)
        same = bool(np.array_equal(x, y))
        assert same, (i, err)


# one tile; tiles of 64 x 64 points; of 64 x 128
@pytest.mark.parametrize("Z,X,S", [(33, 81, 1), (121, 200, 12), (130, 310, 12)])
def test_gradient_of_a2_alone_equals_one_step_kernels(monkeypatch, Z, X, S):
    from adfwi_amd.propagator import acoustic_kernels as ak
    out = []
    for fuse in ("0", "1"):
        monkeypatch.setenv("ADFWI_FUSE_STEPS", fuse)
        rng = np.random.default_rng(Z * 1000 + X)
        rx = np.arange(0, X - 1, 2)
        gen = torch.Generator().manual_seed(Z + X)
        g = ak.AcousticGeometry(Z, X, 37, False, 1, rng.integers(1, Z - 1, S), rng.integers(1, X - 1, S),
                                np.full(len(rx), 2), rx, DEV, resident_images=1)
        field = lambda a, b: (a + (b - a) * torch.rand((Z, X), generator=gen)).to(DEV)
        a1, a2, omk = field(0.1, 0.3), field(0.1, 0.3), [field(0.9, 1.0) for _ in range(3)]
        src = torch.randn((S, 37), generator=gen).to(DEV)
        x2 = a2.clone().requires_grad_(True)
        res = ak.AcousticWave.apply(a1, x2, src, *omk, g, 12, 11)
        adj = [torch.randn(r.shape, generator=torch.Generator().manual_seed(i)).to(DEV) for i, r in enumerate(res[:3])]
        torch.autograd.backward(res[:3], adj)
        out.append(([r.detach().cpu().numpy() for r in res[:3]], x2.grad.cpu().numpy()))
    for i in range(3):
        assert np.array_equal(out[1][0][i], out[0][0][i]), ("record", i)
    err = rel_l2(out[1][1], out[0][1])
    assert np.abs(out[0][1]).max() > 0 and err <= 5e-6, err
