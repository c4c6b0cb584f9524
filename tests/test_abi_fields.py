"""The C ABI as callers built against earlier headers of the same version use it (host only, no GPU:
calls of zero steps launch nothing)."""
import ctypes
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


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


def test_elastic_forward_ignores_its_reserved_field():
    from adfwi_amd import _native as nat
    at = next(f[0] for f in nat.ElasticFwdArgs._fields_
              if getattr(nat.ElasticFwdArgs, f[0]).offset == nat.ElasticFwdArgs.nsteps.offset + 4)
    fake = 0x1000
    d, a = _desc(3, 60, 90), nat.ElasticFwdArgs()
    for f in ("coef", "src", "src_m", "src_z", "src_x", "pml_x", "pml_z"):
        setattr(d, f, fake)
    a.state_in, a.trace, a.nsteps = fake, fake, 0
    for value in (0, 1, -1):     # a trace of states needs no work buffers
        setattr(a, at, value)
        assert nat.load().adfwi_elastic_forward(ctypes.byref(d), ctypes.byref(a), None) == 0, nat.load().adfwi_last_error()


@pytest.mark.parametrize("name,variant", [("adfwi_acoustic_forward", "sum"), ("adfwi_acoustic_adjoint", "sum"),
                                          ("adfwi_elastic_forward", "totals"), ("adfwi_elastic_adjoint", "totals")])
def test_a_fault_injected_into_an_entry_point_reaches_its_variants(name, variant):
    code = ("from adfwi_amd import _native as nat; lib = nat.load(); "
            f"print(lib.{name}(None, None, None), lib.{name}_{variant}(None, None, None))")
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True,
                         env=dict(os.environ, ADFWI_FAULT_INJECT=name), cwd=ROOT)
    assert out.stdout.split() == ["-4", "-4"], out.stderr
