"""GPU parity at transform lengths with prime factors 7, 11 and 13, which run mixed-radix butterflies of
those radices (2-D up to 2048, 3-D up to 512) instead of Bluestein's identity.

Bounds as at every other length: relative L2 <= 1e-4 against the FP64 oracle, dot test <= 1e-5.
Lengths beyond those limits stay refused.
"""
import numpy as np
import pytest

import oracle as O
import seiswem
from conftest import rel_l2
from test_gpu_bluestein import DOT_TOL, TOL, case
from test_gpu_parity import oparams
from test_gpu_parity3d import dot_test, pspi3d, small3d

pytestmark = pytest.mark.gpu

# nmx, padx -> nkx and its array: the smallest, each radix alone and twice, all three, just under an array
# length and at the 2-D limit
SIZES = [(7, 1), (49, 2), (77, 2), (143, 2), (121, 1), (507, 2), (1001, 2), (1014, 2), (2002, 1)]


@pytest.mark.parametrize("nx,padx", SIZES, ids=[f"nkx{a * b}" for a, b in SIZES])
@pytest.mark.parametrize("pspi,mode", [(False, 0), (True, 0), (True, 1)])
def test_prime_radix_2d(gpu, pspi, mode, nx, padx):
    nz, nt = (20, 128) if nx <= 151 else (8, 64)
    g, vel, wav, rng = case(pspi, nx, padx, nz, nt, seed=nx)
    sx = g.dmx * (nx // 3)
    d = rng.standard_normal((g.nm, g.nt)).astype(np.float32)
    m = rng.standard_normal((g.nm, g.nz)).astype(np.float32)
    kw = dict(vel=vel, wav=wav, geom=g, sx=[sx], pspi_mode=mode)
    e1 = rel_l2(seiswem.ShotProfileWEM(d[None], True, **kw), O.wem(oparams(g, mode), vel, wav, sx, d=d, adj=True))
    e2 = rel_l2(seiswem.ShotProfileWEM(m, False, **kw)[0], O.wem(oparams(g, mode), vel, wav, sx, m=m, adj=False))
    print(f"pspi={pspi} mode={mode} nkx={nx * padx}: migrate {e1:.3e} model {e2:.3e}", flush=True)
    assert e1 <= TOL and e2 <= TOL


@pytest.mark.parametrize("nx,ny,nz", [(77, 39, 10), (35, 143, 8), (242, 22, 6)], ids=["154x78", "70x286", "484x44"])
def test_prime_radix_3d(gpu, nx, ny, nz):
    for make in (small3d, pspi3d):
        g, vel, refl, wav, sx, sy = make(nx, ny, nz)
        d = np.random.default_rng(nx).standard_normal((g.nm, g.nt)).astype(np.float32)
        o = (oparams(g), vel, wav, float(sx[0]), float(sy[0]))
        kw = dict(vel=vel, wav=wav, geom=g, sx=sx, sy=sy)
        e1 = rel_l2(seiswem.ShotProfileWEM(d[None], True, **kw), O.wem(*o, d=d, adj=True))
        e2 = rel_l2(seiswem.ShotProfileWEM(refl, False, **kw)[0], O.wem(*o, m=refl, adj=False))
        print(f"{nx}x{ny} pspi={g.pspi}: migrate {e1:.3e} model {e2:.3e}", flush=True)
        assert e1 <= TOL and e2 <= TOL


def test_prime_radix_3d_dot(gpu):
    g, vel, refl, wav, sx, sy = small3d(39, 77, 12)
    assert dot_test(g, vel, wav, sx, sy, 9)[2] <= DOT_TOL


@pytest.mark.parametrize("nx,ny", [(1092, 1), (64, 273)], ids=["2d_nkx2184", "3d_nky546"])
def test_prime_radix_beyond_the_limits_is_refused(gpu, nx, ny):
    g = seiswem.WemGeometry(nt=64, dt=0.004, nmx=nx, dmx=10.0, nmy=ny, dmy=10.0, nz=4, dz=10.0, pspi=False)
    vel = np.full((g.nm, 4), 2000.0, np.float32)
    with pytest.raises(seiswem.SwemError) as e:
        seiswem.Plan(g, vel, np.ones(64, np.float32))
    assert e.value.code == seiswem.SWEM_EUNSUPPORTED
