"""One elastic geometry used for models with and without C15 / C35: its buffer sizes do not depend on
which, and a call for one kind leaves the geometry of a pending backward pass of the other alone."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import ELASTIC_NAMES, elastic_random_case


@pytest.mark.parametrize("damping,nn", [(0, 2), (1, 2), (0, 3), (1, 5)])
@pytest.mark.parametrize("Z,X", [(9, 9), (122, 240), (182, 361), (362, 1040)])
@pytest.mark.parametrize("S", [1, 4, 8, 33])
def test_layout_does_not_depend_on_aniso(S, Z, X, damping, nn):
    from adfwi_amd import _native as nat
    lib, out = nat.load(), []
    for aniso in (0, 1):
        d, L = nat.ElasticDesc(), nat.Layout()
        d.abi_version, d.struct_size = nat.ABI_VERSION, ctypes.sizeof(nat.ElasticDesc)
        d.nshots, d.nz, d.nx, d.pitch = S, max(Z, 2 * nn + 5), max(X, 2 * nn + 5), -(-max(X, 2 * nn + 5) // 64) * 64
        d.nt, d.nrec, d.aniso, d.damping, d.nn = 10, 0, aniso, damping, nn
        assert lib.adfwi_elastic_get_layout(ctypes.byref(d), ctypes.byref(L)) == 0
        out.append([getattr(L, f[0]) for f in nat.Layout._fields_])
    assert out[0] == out[1]


def _geometry(g, m, aniso):
    from adfwi_amd.propagator.elastic_kernels import ElasticGeometry
    half = torch.tensor(g["mt"]) / 2
    src_m = torch.stack([-half[:, 0, 0], -half[:, 2, 2], -half[:, 0, 2]], dim=1)
    zoff = m["nabc"] + 2
    return ElasticGeometry(m["nz"] + zoff + m["nabc"], m["nx"] + 2 * m["nabc"], m["nt"], False, g["src_z"] + zoff,
                           g["src_x"] + m["nabc"], src_m, g["rcv_z"] + zoff, g["rcv_x"] + m["nabc"], "cuda:0",
                           aniso=aniso)


@pytest.mark.gpu
@pytest.mark.parametrize("built_for", [False, True])
def test_one_geometry_for_models_with_and_without_c15_c35(built_for):
    """122 x 240 points, 8 shots: eight sets of gradient planes on tiles, two in the step kernels.  The
    kernels and the order of their sums are those of a geometry of the call's own: the same bits."""
    from test_elastic_gpu import _dropin, _loss
    cases = [elastic_random_case(104, 224, 8, 13, 8, False, seed=41, aniso=aniso) for aniso in (False, True)]
    alone = []
    for g, m in cases:
        res, leaves, w = _dropin(g, m, want_grad=True)
        _loss(res, g["weights"]).backward()
        alone.append((res, leaves, w))
    geom = _geometry(*cases[0], built_for)
    runs = [_dropin(g, m, want_grad=True, geometry=geom) for g, m in cases]   # both forwards, then both backwards
    for (g, _), (res, _, _) in zip(cases, runs):
        _loss(res, g["weights"]).backward()
    torch.cuda.synchronize()
    assert geom.aniso == built_for
    for (ra, la, wa), (rb, lb, wb) in zip(alone, runs):
        for k in ELASTIC_NAMES:
            assert torch.equal(ra[k], rb[k]), k
        for k in la:
            assert la[k].grad.abs().max() > 0 and torch.equal(la[k].grad, lb[k].grad), k
        assert torch.equal(wa.grad, wb.grad)
