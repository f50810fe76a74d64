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


def _migrate(nx, nz):
    g, vel, wav = _case(nx=nx, nz=nz)
    rng = np.random.default_rng(nx + nz)
    d = rng.standard_normal((1, g.nm, g.nt)).astype(np.float32)
    m = seiswem.ShotProfileWEM(d, True, vel=vel, wav=wav, geom=g, sx=[100.0])
    return g, vel, wav, d, m


def test_host_calls_keep_and_give_back(gpu):
    """Host calls of alternating sizes, each on blocks that others have written: the image of a resident plan,
    bit for bit.  What they keep goes by release_memory and before a plan is created."""
    sizes = [(256, 400), (64, 20), (256, 390), (250, 400), (128, 100), (256, 400)]
    images = [_migrate(nx, nz) for nx, nz in sizes]
    # the phase tables of the last call: 400 depths x 153 frequencies x (257 wavenumbers + 256 traces) x 8 bytes
    tables = 400 * 153 * (257 + 256) * 8
    kept = _used()
    seiswem.release_memory()
    assert kept - _used() >= tables
    for g, vel, wav, d, m in images:
        plan = seiswem.Plan(g, vel, wav)
        ref = plan.migrate(seiswem.DeviceArray(d.shape, d), [100.0]).download()
        plan.close()
        assert np.array_equal(m, ref) and np.any(m)
    _migrate(256, 400)
    g, vel, wav = _case()
    kept = _used()
    plan = seiswem.Plan(g, vel, wav)
    assert kept - _used() >= tables - 32 * MIB  # the new plan's own buffers are smaller than that
    plan.close()


def test_release_memory_refuses_a_negative_device(gpu):
    with pytest.raises(seiswem.SwemError) as e:
        seiswem.release_memory(-1)
    assert e.value.code == seiswem.SWEM_EINVAL
    seiswem.release_memory(63)  # nothing kept there
