"""The acoustic tile kernels (up to four steps per launch on register tiles) against the one-step
kernels with separate gather and inject launches (ADFWI_FUSE_STEPS=0): records, and the wavelet
gradient, bit for bit; energy maps and the A1 / A2 gradients, whose terms are added in another
order, to rounding.

The grids pick every tile shape (40 x 64, 64 x 64 and 64 x 128 points, which store 16 x 40, 40 x 40
and 40 x 104) and put the grid's edges at, one short of and one past a tile's; odd widths leave a
lane with one column; one grid is the smallest the library takes.  nt and the checkpoint interval
leave launches of one, two, three and four steps.

Tolerance of the reordered sums: N = shots * steps terms per point, each addition rounding to 2^-24:
sqrt(N) * 2^-24 for terms of one sign (the energy maps), 2.9e-6 for 64 shots; 5e-6, and for more shots
twice that bound, leaves room for the gradients' cancellation.
"""
import numpy as np
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # Z, X, shots, free-surface row (0: none)
    (8, 8, 1, 0),            # smallest
    (33, 81, 2, 0),          # one past two small tiles each way
    (48, 80, 1, 8),          # small tiles ending at the edges of the grid, free surface
    (121, 200, 12, 0),       # 64 x 64 tiles: 4 x 5 x 12 = 240
    (120, 161, 15, 10),      # 3 x 5 x 15 with a free surface
    (41, 105, 64, 0),        # 64 x 128 tiles, one past a tile each way
    (40, 208, 63, 6),        # 64 x 128 tiles ending at the grid's edges
    (79, 103, 64, 0),        # odd width, last tile one column short
    (41, 105, 81, 0),        # over 256 workgroups: pairs of shots, the last group one shot
    (41, 105, 161, 5),       # groups of three, the last of two
]


@pytest.mark.parametrize("needs", ["a1", "all"])
@pytest.mark.parametrize("Z,X,S,fs", CASES)
def test_tiles_equal_one_step_kernels(monkeypatch, Z, X, S, fs, needs):
    from adfwi_amd.propagator import acoustic_kernels as ak
    rng = np.random.default_rng(Z * 1000 + X)
    tol = max(5e-6, 2 * (S * 37) ** 0.5 * 2 ** -24 if S > 64 else 0)
    nt, k = 37, 11                       # segments of 11: launches of 4, 4 and 3 steps; the last of 4
    nabc = fs if fs else 1
    lo = max(fs, 1)
    src_z, src_x = rng.integers(lo, Z - 1, S), rng.integers(1, X - 1, S)
    src_z[0], src_x[0] = lo, X - 2       # on the edges of the grid
    # receivers: a line along a row, a second row and points on tile edges
    pts = {(lo + 1, x) for x in range(0, X - 1, 2)} | {(Z // 2, x) for x in range(0, X - 1, 5)}
    pts |= {(min(z, Z - 2), min(x, X - 2)) for z in (15, 16, 39, 40) for x in (39, 40, 103, 104)}
    pts = np.array(sorted(p for p in pts if p[0] != fs - 1))
    gen = torch.Generator().manual_seed(Z + X)
    field = lambda a, b: (a + (b - a) * torch.rand((Z, X), generator=gen)).to(DEV)
    a1, a2 = field(0.1, 0.3), field(0.1, 0.3)
    omk = [field(0.9, 1.0) for _ in range(3)]
    src = torch.randn((S, nt), generator=gen).to(DEV)
    outs = []
    for fuse in ("0", "1"):
        monkeypatch.setenv("ADFWI_FUSE_STEPS", fuse)
        g = ak.AcousticGeometry(Z, X, nt, bool(fs), nabc, src_z, src_x, pts[:, 0], pts[:, 1], DEV, resident_images=1)
        assert g.tiled == (fuse == "1")
        x1, x2, w = a1.clone().requires_grad_(True), a2.clone().requires_grad_(needs == "all"), src.clone()
        w.requires_grad_(needs == "all")
        res = ak.AcousticWave.apply(x1, x2, w, *omk, g, nt // 3, k)
        nrec = 3 if needs == "all" else 1
        gr = [torch.randn(r.shape, generator=torch.Generator().manual_seed(i)).to(DEV) for i, r in enumerate(res[:nrec])]
        torch.autograd.backward(res[:nrec], gr)
        torch.cuda.synchronize()
        outs.append(([r.detach().cpu().numpy() for r in res], x1.grad.cpu().numpy(),
                     None if x2.grad is None else x2.grad.cpu().numpy(), None if w.grad is None else w.grad.cpu().numpy()))
    (r0, g0, h0, w0), (r1, g1, h1, w1) = outs
    for i in range(3):
        assert np.array_equal(r0[i], r1[i]), ("record", i, rel_l2(r1[i], r0[i]))
    for i in range(3, 6):
        assert rel_l2(r1[i], r0[i]) <= tol, ("energy", i, rel_l2(r1[i], r0[i]))
    assert rel_l2(g1, g0) <= tol, rel_l2(g1, g0)
    if needs == "all":
        assert rel_l2(h1, h0) <= tol, rel_l2(h1, h0)
        assert np.array_equal(w0, w1), rel_l2(w1, w0)
