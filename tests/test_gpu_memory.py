"""Device memory across plans and host calls."""
import numpy as np
import pytest
import torch

import seiswem
from seiswem import synth

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def _case(nt=500, nz=20, nx=64):
    g = seiswem.WemGeometry(nt=nt, dt=0.004, nmx=nx, dmx=10.0, nz=nz, dz=10.0, fmin=2.0, fmax=40.0, pspi=False)
    vel = np.full((nx, nz), 2000.0, np.float32)
    return g, vel, synth.wavelet_trace(nt, g.dt, 20.0)


def _used():
    free, total = torch.cuda.mem_get_info()
    return total - free


def test_plans_leave_nothing(gpu):
    """A plan built and closed leaves no device memory: the angle table of its Fourier bases (2 ntfft + nf
    doubles, 130 KiB here) goes with it."""
    g, vel, wav = _case(nt=4000, nz=2)
    seiswem.Plan(g, vel, wav).close()
    before = _used()
    for _ in range(160):
        seiswem.Plan(g, vel, wav).close()
    assert _used() - before <= 4 * MIB  # 20 MiB of tables, were they left
