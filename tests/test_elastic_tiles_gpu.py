"""The elastic tile kernels (up to two steps per launch on register tiles, a trace of five totals)
against the one-step kernels (explicit tiling, a trace of the ten splits): records, checkpoints,
final states and the wavelet gradient are formed by the same operations in the same order, so they
are equal bit for bit; the terms of the coefficient gradients are added in another order.

The grids pick every tile height (32, 48 and 64 rows, which store 20, 36 and 52) and end at, one
short of and one past a tile's edge each way (52 columns, from the window's first); one grid is the
smallest the library takes; steps and checkpoint cuts leave launches of one and of two steps.  The
adjoint takes 32 rows and single shots in the first five, 48 rows and groups of 1, 2 and more shots,
the last of them smaller, in the others.

Tolerance of the reordered sums: N = shots * steps terms per point, at most 80 * 13 = 1040, each
addition rounding to 2^-24: sqrt(N) * 2^-24 = 1.9e-6; 5e-6 leaves room for cancellation.
"""
import numpy as np
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # Z, X, shots, free surface, vertical force
    (9, 9, 1, False, False),       # smallest
    (9, 9, 2, True, False),
    (24, 56, 3, True, True),       # one tile of 20 x 52, filled
    (25, 57, 3, True, False),      # one past it
    (63, 107, 2, False, True),     # one short of 3 x 2 tiles
    (76, 160, 30, True, False),    # 48 rows: 2 x 3 tiles, filled (4 x 3 x 30 of 32 rows are over 256)
    (77, 109, 28, False, False),   # 48 rows: 3 x 3 tiles, one past
    (108, 108, 61, True, False),   # 64 rows: 2 x 2 tiles, filled
    (64, 60, 80, True, True),      # more tiles than compute units at every height: 32 rows
]


# three-term differences (6th to 10th order, one step per launch): the same edges
CASES3 = [
    # Z, X, shots, free surface, vertical force, half-order
    (11, 11, 1, False, False, 3),  # smallest
    (15, 15, 2, True, False, 5),
    (26, 58, 3, True, True, 3),    # one tile of 20 x 52, filled
    (29, 61, 3, True, False, 4),   # one past it
    (68, 112, 2, False, True, 5),  # two short of 3 x 2 tiles
    (78, 162, 30, True, False, 3), # 48 rows, filled
    (110, 110, 61, True, False, 3),  # 64 rows, filled
    (66, 62, 80, False, True, 3),  # 64 rows, more tiles than compute units
]


@pytest.mark.parametrize("Z,X,S,fs,force", CASES)
def test_tiles_equal_one_step_kernels(Z, X, S, fs, force):
    _compare(Z, X, S, fs, force, 2)


@pytest.mark.parametrize("Z,X,S,fs,force,nn", CASES3)
def test_three_term_tiles_equal_one_step_kernels(Z, X, S, fs, force, nn):
    _compare(Z, X, S, fs, force, nn)


@pytest.mark.parametrize("Z,X,S,fs,force,nn", [c + (2,) for c in CASES if c[2] != 80] + CASES3[:5] + [
    (24, 52, 3, True, True, 2),    # one tile of 20 x 48, filled
    (25, 53, 3, True, True, 2),    # one past it
    (64, 60, 140, True, False, 2),  # more tiles than compute units at every height: 32 rows
    (66, 62, 80, True, True, 3),
])
def test_damping_tiles_equal_one_step_kernels(Z, X, S, fs, force, nn):
    _compare(Z, X, S, fs, force, nn, damping=True)


def test_three_term_tiles_end_at_three_rounds():
    from adfwi_amd.propagator import elastic_kernels as ek
    for S, tiled in ((192, True), (193, False)):   # 2 x 2 tiles of 52 x 52 each
        one = np.full(S, 9)
        g = ek.ElasticGeometry(66, 62, 4, True, one, one, torch.zeros(S, 3), one[:1], one[:1], DEV, nn=3)
        assert g.tiled == tiled


def _compare(Z, X, S, fs, force, nn, damping=False):
    from adfwi_amd.propagator import elastic_adjoint as ea
    from adfwi_amd.propagator import elastic_kernels as ek
    rng = np.random.default_rng(Z * 1000 + X)
    nt, k = 13, 5                                   # segments of 5, 5 and 3 steps
    src_z, src_x = rng.integers(nn, Z - nn, S), rng.integers(nn, X - nn, S)
    src_z[0], src_x[0] = nn, X - nn - 1                   # on the window's corner
    # a line along row nn+1, points on tile edges, the window's last row and column
    w = lambda z, x: (min(z, Z - nn - 1), min(x, X - nn - 1))
    pts = {w(nn + 1, x) for x in range(nn, X - nn, 3)} | {(nn, nn), w(Z, X)}
    pts |= {w(nn + z, nn + x) for z in (19, 20, 35, 36, 51, 52) for x in (51, 52)}
    pts = np.array(sorted(pts))
    gen = torch.Generator().manual_seed(Z + X)
    rand = lambda a, b, *shape: a + (b - a) * torch.rand(shape, generator=gen)
    src_m, src_fz = rand(-1, 1, S, 3), rand(-1, 1, S) if force else None
    coef_fields = [rand(a, b, Z, X).to(DEV) for a, b in ((5, 9), (1, 3), (5, 9), (1, 3), (.3, .6), (.3, .6))]
    bcx, bcz = rand(0, 20, 1, X).expand(Z, X), rand(0, 20, Z, 1).expand(Z, X)
    taper = rand(0.9, 1.0, Z, X).to(DEV)
    src = torch.randn((S, nt), generator=gen).to(DEV)
    scalars = (1e-2, 2e-2, 2.5e-2, 0.5, 0.4) + ((1.125, -1.0 / 24) if nn == 2 else (75.0 / 64, -25.0 / 384))
    out = []
    for tile_z in (0, 8):   # three-term: c2 = 3 / 640
        g = ek.ElasticGeometry(Z, X, nt, fs, src_z, src_x, src_m, pts[:, 0], pts[:, 1], DEV, tile_z=tile_z,
                               shots_per_wave=int(tile_z > 0), src_fz=src_fz, nn=nn, c2=0.0 if nn == 2 else 3.0 / 640,
                               damping=damping)
        assert g.tiled == (tile_z == 0)
        px, pz = (t.to(DEV) for t in ek.pml_factors(bcx, bcz, scalars[0], g.pitch))
        coef = g.pack_coef(coef_fields + [None, None])
        damp = g.pack_plane(taper) if damping else None
        out.append((g, coef, px, pz, damp, ek.run_forward(g, coef, px, pz, src, scalars, ckpt_every=k, damp=damp)))
    (g, coef, px, pz, damp, a), b = out[0], out[1][5]
    torch.cuda.synchronize()
    for i in range(5):
        assert torch.isfinite(b["rec"][i]).all() and b["rec"][i].abs().max() > 0
        assert torch.equal(a["rec"][i], b["rec"][i]), ("record", i, rel_l2(a["rec"][i].cpu(), b["rec"][i].cpu()))
    assert torch.equal(a["ckpt"], b["ckpt"]) and torch.equal(a["final"], b["final"])
    g_rec = [torch.randn((S, nt, len(pts)), generator=gen).to(DEV) for _ in range(5)]
    needs = [True] * 6 + [False] * 2 + [True]
    if damping:   # the trace is the state's five fields with either kernel
        grads = [ea.run_backward(x[0], coef, src, px, pz, scalars, x[5]["ckpt"], k, g_rec, needs, damp=x[4]) for x in out]
    else:
        grads = [ea.run_backward(g, coef, src, px, pz, scalars, a["ckpt"], k, g_rec, needs, totals=totals)
                 for totals in (True, False)]
    torch.cuda.synchronize()
    for i in range(6):
        assert grads[1][0][i].abs().max() > 0
        err = rel_l2(grads[0][0][i].cpu().numpy(), grads[1][0][i].cpu().numpy())
        assert err <= 5e-6, ("gradient", i, err)
    assert torch.equal(grads[0][1], grads[1][1])
