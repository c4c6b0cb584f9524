"""A device time base that takes a window over the ends of the run: the steps inside [0, nt) are
taken, as one by one from the same state, the others skipped."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _problem(nt, window):
    from adfwi_amd import _native as nat
    from adfwi_amd.propagator.acoustic_kernels import AcousticGeometry
    Z, X, S = 48, 120, 3
    gen = torch.Generator().manual_seed(nt)
    rx = np.arange(0, X - 1, 3)
    g = AcousticGeometry(Z, X, nt, False, 1, np.full(S, 9), np.array([20, 60, 90]), np.full(len(rx), 7), rx, DEV)
    field = lambda a, b: (a + (b - a) * torch.rand((Z, X), generator=gen)).to(DEV)
    coef = g.pack_coef(field(0.9, 1.0), field(0.1, 0.3), field(0.9, 1.0), field(0.1, 0.3), field(0.9, 1.0))
    src = torch.randn((S, nt), generator=gen).to(DEV)

    def run(base, state, energy, rec):
        """One window of steps base, base + 1, ...; returns the state after it."""
        work = torch.zeros_like(g.state(2))
        tb = torch.tensor([base], dtype=torch.int32, device=DEV)
        d, a = g.desc(coef, src), nat.AcousticFwdArgs()
        a.state_in = state.data_ptr()
        a.work[0], a.work[1] = work[0].data_ptr(), work[1].data_ptr()
        a.t0, a.nsteps, a.energy_u_from, a.t_base, a.fuse_steps = 0, window, 1, tb.data_ptr(), g.fuse_steps
        a.energy = energy.data_ptr()
        a.rec_p, a.rec_u, a.rec_w = (r.data_ptr() for r in rec)
        a.rcv_map = g.rcv_map.data_ptr()
        nat.check(nat.load().adfwi_acoustic_forward(ctypes.byref(d), ctypes.byref(a), nat.stream_handle(src.device)),
                  "adfwi_acoustic_forward")
        torch.cuda.synchronize()
        return work[0] if a.state_out == work[0].data_ptr() else work[1]
    return g, coef, src, run


@pytest.mark.parametrize("nt,window", [(10, 8), (11, 8), (13, 4), (13, 12)])
def test_last_window_takes_its_steps_inside_the_run(nt, window):
    from adfwi_amd.propagator.acoustic_kernels import run_forward
    g, coef, src, run = _problem(nt, window)
    ref = run_forward(g, coef, src, energy_u_from=1)
    rec = [torch.zeros((g.S, nt, g.R), device=DEV) for _ in range(3)]
    energy = torch.zeros((int(g.layout.ngroups), 2, g.Z, g.pitch), device=DEV)
    state = g.state()[0]
    for base in range(0, nt, window):
        state = run(base, state, energy, rec)
    for i in range(3):
        assert ref["rec"][i].abs().max() > 0 and torch.equal(rec[i], ref["rec"][i]), i
    # the launches cut the sums of at most 13 terms differently: sqrt(13) * 2^-24 = 2.1e-7
    e = energy.sum(0)[:, :, :g.X]
    for i in range(2):
        assert (e[i] - ref["energy"][i]).norm() <= 1e-6 * ref["energy"][i].norm(), i


def test_window_before_the_run_takes_its_steps_inside_it():
    from adfwi_amd.propagator.acoustic_kernels import run_forward
    g, coef, src, run = _problem(10, 8)
    ref = run_forward(g, coef, src, energy_u_from=None)
    rec = [torch.zeros((g.S, 10, g.R), device=DEV) for _ in range(3)]
    run(-2, g.state()[0], torch.zeros((int(g.layout.ngroups), 2, g.Z, g.pitch), device=DEV), rec)
    for i in range(3):
        assert torch.equal(rec[i][:, :6], ref["rec"][i][:, :6]) and not rec[i][:, 6:].any(), i
