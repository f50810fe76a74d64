"""GPU parity at power-of-two transform lengths around 2 nmx = nkx, where the march kernels switch to the
forms that drop the zero half of every line: pad factor 1 (all points live: the general form), 2 (exactly
half of them) and 4 (a quarter).

Bound as at every other size: relative L2 <= 1e-4 against the FP64 oracle.
"""
import numpy as np
import pytest

import oracle as O
import seiswem
from conftest import rel_l2
from test_gpu_bluestein import TOL, case
from test_gpu_parity import oparams
from test_gpu_parity3d import pspi3d, small3d

pytestmark = pytest.mark.gpu


def both(g, vel, wav, sx, sy, d, m, mode):
    kw = dict(vel=vel, wav=wav, geom=g, sx=[sx], sy=[sy], pspi_mode=mode)
    op = oparams(g, mode)
    op.nmy, op.dmy = g.nmy, g.dmy
    e1 = rel_l2(seiswem.ShotProfileWEM(d[None], True, **kw), O.wem(op, vel, wav, sx, sy, d=d, adj=True))
    e2 = rel_l2(seiswem.ShotProfileWEM(m, False, **kw)[0], O.wem(op, vel, wav, sx, sy, m=m, adj=False))
    return e1, e2


@pytest.mark.parametrize("nx,ny,padx", [(128, 128, 1), (256, 128, 1), (64, 128, 2), (256, 64, 2), (32, 64, 4), (128, 32, 4)])
@pytest.mark.parametrize("pspi,mode", [(False, 0), (True, 0), (True, 1)])
def test_half_lines_3d(gpu, pspi, mode, nx, ny, padx):
    g, vel, refl, wav, sx, sy = (pspi3d if pspi else small3d)(nx, ny, 6)
    g.padx = padx
    d = np.random.default_rng(nx + padx).standard_normal((g.nm, g.nt)).astype(np.float32)
    e1, e2 = both(g, vel, wav, float(sx[0]), float(sy[0]), d, refl, mode)
    print(f"{nx}x{ny} padx={padx} pspi={pspi} mode={mode}: migrate {e1:.3e} model {e2:.3e}", flush=True)
    assert e1 <= TOL and e2 <= TOL


@pytest.mark.parametrize("nx,padx", [(128, 1), (512, 1), (64, 2), (512, 2), (32, 4), (256, 4)])
@pytest.mark.parametrize("pspi,mode", [(False, 0), (True, 0), (True, 1)])
def test_half_lines_2d(gpu, pspi, mode, nx, padx):
    g, vel, wav, rng = case(pspi, nx, padx, 8, 64, seed=nx)
    d = rng.standard_normal((g.nm, g.nt)).astype(np.float32)
    m = rng.standard_normal((g.nm, g.nz)).astype(np.float32)
    e1, e2 = both(g, vel, wav, g.dmx * (nx // 3), 0.0, d, m, mode)
    print(f"nkx={nx * padx} padx={padx} pspi={pspi} mode={mode}: migrate {e1:.3e} model {e2:.3e}", flush=True)
    assert e1 <= TOL and e2 <= TOL


@pytest.mark.parametrize("variant", [seiswem.VARIANT_AUTO, seiswem.VARIANT_PAIR, seiswem.VARIANT_PAIR8])
@pytest.mark.parametrize("nx", [256, 512, 1024])
def test_single_steps_before_the_lockstep_ones(gpu, nx, variant):
    """A source below the receivers: the first depths step the receiver alone, the rest both in lockstep
    through the same LDS buffers."""
    g, vel, wav, rng = case(False, nx, 2, 16, 64, seed=nx + 1)
    g.sz = g.oz + 4.5 * g.dz
    d = rng.standard_normal((g.nm, g.nt)).astype(np.float32)
    sx = g.dmx * (nx // 3)
    m = seiswem.ShotProfileWEM(d[None], True, vel=vel, wav=wav, geom=g, sx=[sx], variant=variant)
    err = rel_l2(m, O.wem(oparams(g), vel, wav, sx, d=d, adj=True))
    print(f"nkx={2 * nx} variant={variant}: migrate {err:.3e}", flush=True)
    assert err <= TOL
