"""The per-trace L2 kernel with 8, 16 and 32 receivers per workgroup (up to two workgroups per CU, and
more) against the same formulas in float64: trace counts one short of, at and one past a group's, fewer
samples than a workgroup takes side by side, one, and some that leave a remainder; maxima that occur
twice, whose gradient goes to the first.

Tolerance: a residual n - b of operands of order one carries at most 2 * 2^-24 of them; sums over
nt <= 600 samples add (600 / 32 + 6 + 16) roundings of 2^-24 each, 2.5e-6 for terms all rounded one
way; their square root halves that.  4e-6.
"""
import numpy as np
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = 4e-6


@pytest.mark.parametrize("flags", [0, 1, 2, 3])
@pytest.mark.parametrize("S,nt,R", [
    (1, 1, 1), (3, 127, 7), (2, 129, 8), (2, 600, 9),          # 8 receivers per workgroup
    (512, 40, 8), (64, 129, 65),                               # (the last group of 8; 9 groups of 8: 16)
    (300, 65, 16), (257, 64, 17),                              # 16; 17 takes two groups of 16: 32
    (1030, 33, 31), (600, 32, 33),                             # 32
])
def test_trace_l2_groups(S, nt, R, flags):
    from adfwi_amd.fwi.misfit import _trace_l2
    gen = torch.Generator().manual_seed(S * 1000 + nt + R)
    a, b = (torch.randn((S, nt, R), generator=gen) for _ in range(2))
    a[0, nt // 2, 0] = 5.0
    a[0, nt - 1, 0] = -5.0                    # an equal maximum later in time
    dt = 1e-3
    loss, ga, gb = _trace_l2(a.to(DEV), b.to(DEV), dt, flags, True, True)
    x, y = a.double(), b.double()
    m, ts = x.abs().max(dim=1, keepdim=True)  # (the CPU's max takes the first)
    assert ts[0, 0, 0] == nt // 2 or nt == 1
    n = x / m if flags & 1 else x
    rsd = n - y
    e = (rsd ** 2 * dt).sum(1, keepdim=True)
    w = torch.full_like(e, dt) if flags & 2 else dt / e.sqrt()
    g = w * rsd
    ref = g
    if flags & 1:
        ref = g / m
        q = (rsd * x).sum(1, keepdim=True)
        ref = ref.scatter_add(1, ts, -(x.gather(1, ts).sign() * w * q / m ** 2))
    want = (0.5 * e if flags & 2 else e.sqrt())[:, 0]
    for got, exp in ((loss, want), (ga, ref), (gb, -g)):
        if nt == 1 and flags & 1 and got is ga:
            continue                          # one sample: n is its sign, the exact gradient is zero
        err = rel_l2(got.cpu().numpy(), exp.numpy())
        assert err <= TOL, err
