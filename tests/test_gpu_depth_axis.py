"""Depth axes that run upward (dz < 0), source and receivers inside them: the lockstep steps of the split-step
pair kernel come first, then one wavefield steps alone through the same LDS buffers, or neither does.

Bound as at every other size: relative L2 <= 1e-4 against the FP64 oracle.
"""
import numpy as np
import pytest

import oracle as O
import seiswem
from conftest import rel_l2
from test_gpu_bluestein import TOL, case
from test_gpu_ewem import case as ecase
from test_gpu_ewem import TOL as ETOL
from test_gpu_ewem import run
from test_gpu_parity import oparams

pytestmark = pytest.mark.gpu
LEVELS = [(95.0, 65.0), (65.0, 95.0), (95.0, 95.0)]  # source, receivers: depths 150, 140 .. 0


def _upward(g):
    g.oz, g.dz = 150.0, -10.0


@pytest.mark.parametrize("variant", [seiswem.VARIANT_AUTO, seiswem.VARIANT_PAIR, seiswem.VARIANT_PAIR8])
@pytest.mark.parametrize("sz,gz", LEVELS)
@pytest.mark.parametrize("nx,padx", [(64, 2), (128, 2), (512, 1), (1024, 1), (512, 2), (1024, 2)])
def test_split_step(gpu, nx, padx, sz, gz, variant):
    g, vel, wav, rng = case(False, nx, padx, 16, 64, seed=nx + 2)
    _upward(g)
    g.sz, g.gz = sz, gz
    d = rng.standard_normal((g.nm, g.nt)).astype(np.float32)
    sx = g.dmx * (nx // 3)
    m = seiswem.ShotProfileWEM(d[None], True, vel=vel, wav=wav, geom=g, sx=[sx], variant=variant)
    err = rel_l2(m, O.wem(oparams(g), vel, wav, sx, d=d, adj=True))
    print(f"nkx={nx * padx} sz={sz} gz={gz} variant={variant}: migrate {err:.3e}", flush=True)
    assert np.any(m) and err <= TOL


@pytest.mark.parametrize("sz,gz", LEVELS)
@pytest.mark.parametrize("pspi,mode", [(False, 0), (True, 0), (True, 1)])
@pytest.mark.parametrize("nx", [256, 150])
def test_modelling_and_pspi(gpu, nx, pspi, mode, sz, gz):
    g, vel, wav, rng = case(pspi, nx, 2, 16, 64, seed=nx + 3)
    _upward(g)
    g.sz, g.gz = sz, gz
    sx = g.dmx * (nx // 3)
    kw = dict(vel=vel, wav=wav, geom=g, sx=[sx], pspi_mode=mode)
    op = oparams(g, mode)
    d = rng.standard_normal((g.nm, g.nt)).astype(np.float32)
    m = rng.standard_normal((g.nm, g.nz)).astype(np.float32)
    e1 = rel_l2(seiswem.ShotProfileWEM(d[None], True, **kw), O.wem(op, vel, wav, sx, d=d, adj=True))
    e2 = rel_l2(seiswem.ShotProfileWEM(m, False, **kw)[0], O.wem(op, vel, wav, sx, m=m, adj=False))
    print(f"nkx={2 * nx} pspi={pspi} mode={mode} sz={sz} gz={gz}: migrate {e1:.3e} model {e2:.3e}", flush=True)
    assert e1 <= TOL and e2 <= TOL


@pytest.mark.parametrize("sz,gz", LEVELS)
def test_elastic(gpu, sz, gz):
    g, p, vp, vs, wav, rng = ecase(512, nz=16, nt=128, seed=9)
    for q in (g, p):
        q.oz, q.dz, q.sz, q.gz = 150.0, -10.0, sz, gz
    sx = g.dmx * 170
    ux, uy, uz = rng.standard_normal((3, g.nm, g.nt)).astype(np.float32)
    mpp, _, mps2 = run(g, vp, vs, wav, sx, True, ux, uy, uz)
    rpp, rps2 = O.ewem(p, vp, vs, wav, sx, ux=ux, uz=uz, adj=True)
    errs = [rel_l2(mpp, rpp), rel_l2(mps2, rps2)]
    print(f"sz={sz} gz={gz}: PP {errs[0]:.3e} PS {errs[1]:.3e}", flush=True)
    assert np.any(mpp) and max(errs) <= ETOL
