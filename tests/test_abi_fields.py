"""The C ABI as callers built against earlier headers of the same version use it (host only, no GPU:
calls of zero steps launch nothing)."""
import ctypes

import pytest


def _desc(S, Z, X, damping=0, nn=2):
    from adfwi_amd import _native as nat
    d = nat.ElasticDesc()
    d.abi_version, d.struct_size = nat.ABI_VERSION, ctypes.sizeof(nat.ElasticDesc)
    d.nshots, d.nz, d.nx, d.pitch = S, Z, X, -(-X // 64) * 64
    d.nt, d.nrec, d.damping, d.nn = 10, 0, damping, nn
    return d


@pytest.mark.parametrize("damping,nn", [(0, 2), (1, 2), (0, 3), (1, 4)])
@pytest.mark.parametrize("S,Z,X", [(1, 13, 13), (8, 122, 240), (33, 171, 373), (48, 362, 1040)])
def test_elastic_accumulator_is_ngroups_sets(S, Z, X, damping, nn):
    from adfwi_amd import _native as nat
    d, L = _desc(S, Z, X, damping, nn), nat.Layout()
    assert nat.load().adfwi_elastic_get_layout(ctypes.byref(d), ctypes.byref(L)) == 0
    assert L.accum_floats == L.ngroups * 8 * Z * d.pitch
