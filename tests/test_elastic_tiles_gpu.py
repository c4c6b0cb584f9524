"""The elastic tile kernels (up to two steps per launch on register tiles, a trace of five totals)
against the one-step kernels (explicit tiling, a trace of the ten splits): records, checkpoints,
final states and the wavelet gradient are formed by the same operations in the same order, so they
are equal bit for bit; the terms of the coefficient gradients are added in another order.

The grids pick every tile height (32, 48 and 64 rows, which store 20, 36 and 52) and end at, one
short of and one past a tile's edge each way (52 columns, from column 2); one grid is the smallest
the library takes; steps and checkpoint cuts leave launches of one and of two steps.  The adjoint takes 32 rows and
single shots in the first five, 48 rows and groups of 1, 2 and more shots, the last of them smaller,
in the others.

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


@pytest.mark.parametrize("Z,X,S,fs,force", CASES)
def test_tiles_equal_one_step_kernels(Z, X, S, fs, force):
    from adfwi_amd.propagator import elastic_adjoint as ea
    from adfwi_amd.propagator import elastic_kernels as ek
    rng = np.random.default_rng(Z * 1000 + X)
    nt, k = 13, 5                                   # segments of 5, 5 and 3 steps
    src_z, src_x = rng.integers(2, Z - 2, S), rng.integers(2, X - 2, S)
    src_z[0], src_x[0] = 2, X - 3                   # on the window's corner
    # a line along row 3, points on tile edges, the window's last row and column
    pts = {(min(3, Z - 3), x) for x in range(2, X - 2, 3)} | {(2, 2), (Z - 3, X - 3)}
    pts |= {(min(z, Z - 3), min(x, X - 3)) for z in (21, 22, 37, 38, 53, 54) for x in (53, 54)}
    pts = np.array(sorted(pts))
    gen = torch.Generator().manual_seed(Z + X)
    rand = lambda a, b, *shape: a + (b - a) * torch.rand(shape, generator=gen)
    src_m, src_fz = rand(-1, 1, S, 3), rand(-1, 1, S) if force else None
    coef_fields = [rand(a, b, Z, X).to(DEV) for a, b in ((5, 9), (1, 3), (5, 9), (1, 3), (.3, .6), (.3, .6))]
    bcx, bcz = rand(0, 20, 1, X).expand(Z, X), rand(0, 20, Z, 1).expand(Z, X)
    src = torch.randn((S, nt), generator=gen).to(DEV)
    scalars = (1e-2, 2e-2, 2.5e-2, 0.5, 0.4, 1.125, -1.0 / 24)
    out = []
    for tile_z in (0, 8):
        g = ek.ElasticGeometry(Z, X, nt, fs, src_z, src_x, src_m, pts[:, 0], pts[:, 1], DEV, tile_z=tile_z,
                               shots_per_wave=int(tile_z > 0), src_fz=src_fz)
        assert g.tiled == (tile_z == 0)
        px, pz = (t.to(DEV) for t in ek.pml_factors(bcx, bcz, scalars[0], g.pitch))
        coef = g.pack_coef(coef_fields + [None, None])
        out.append((g, coef, px, pz, ek.run_forward(g, coef, px, pz, src, scalars, ckpt_every=k)))
    (g, coef, px, pz, a), b = out[0], out[1][4]
    torch.cuda.synchronize()
    for i in range(5):
        assert torch.isfinite(b["rec"][i]).all() and b["rec"][i].abs().max() > 0
        assert torch.equal(a["rec"][i], b["rec"][i]), ("record", i, rel_l2(a["rec"][i].cpu(), b["rec"][i].cpu()))
    assert torch.equal(a["ckpt"], b["ckpt"]) and torch.equal(a["final"], b["final"])
    g_rec = [torch.randn((S, nt, len(pts)), generator=gen).to(DEV) for _ in range(5)]
    grads = [ea.run_backward(g, coef, src, px, pz, scalars, a["ckpt"], k, g_rec, [True] * 6 + [False] * 2 + [True],
                             totals=totals) for totals in (True, False)]
    torch.cuda.synchronize()
    for i in range(6):
        assert grads[1][0][i].abs().max() > 0
        err = rel_l2(grads[0][0][i].cpu().numpy(), grads[1][0][i].cpu().numpy())
        assert err <= 5e-6, ("gradient", i, err)
    assert torch.equal(grads[0][1], grads[1][1])
