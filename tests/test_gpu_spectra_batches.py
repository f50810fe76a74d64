"""The time <-> frequency products have two tilings, by the number of rows of a launch (128 x 128 outputs per
workgroup, or 32 x 32 with K split over waves), and one summation order: a shot's image and its modelled
records are the same bits alone (the split form) and in a batch large enough for the tiles.

Sizes at the edges: traces and samples that are no multiples of 8, 32 or 128, K below one segment (128), at
one, and over sixteen of them."""
import numpy as np
import pytest

import seiswem
from seiswem import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nt,shots", [(130, 61, 260), (127, 128, 260), (100, 333, 140), (65, 2101, 70)])
def test_spectra_do_not_depend_on_the_batch(gpu, nx, nt, shots):
    g = seiswem.WemGeometry(nt=nt, dt=0.004, nmx=nx, dmx=10.0, nz=3, dz=10.0, fmin=2.0, fmax=60.0, pspi=False)
    rng = np.random.default_rng(nt)
    vel = synth.blob_velocity(nx, 3, 10.0, 10.0, rng, nblobs=2, v0=2000.0)
    plan = seiswem.Plan(g, vel, synth.wavelet_trace(nt, g.dt, 20.0))
    nf = g.sampling()["ifmax"] - g.sampling()["ifmin"]
    assert -(-shots * nx // 128) * -(-2 * nf // 128) >= 256 > -(-nx // 128) * -(-2 * nf // 128), "both tilings are meant"
    sx = (10.0 * (np.arange(shots) % nx)).astype(np.float32)
    d = rng.standard_normal((shots, nx, nt)).astype(np.float32)
    m = seiswem.DeviceArray((nx, 3), rng.standard_normal((nx, 3)))
    images = plan.migrate_each(seiswem.DeviceArray(d.shape, d), sx).download()
    records = plan.model(m, sx).download()
    for s in (0, 1, shots // 2, shots - 1):
        one = plan.migrate_each(seiswem.DeviceArray((1, nx, nt), d[s]), sx[s:s + 1]).download()[0]
        assert np.array_equal(one, images[s]) and np.any(one)
        assert np.array_equal(plan.model(m, sx[s:s + 1]).download()[0], records[s])
    plan.close()
