"""3-D PSPI with SWEM_PREC_FP32 (the reference's float kz phases, wem.c:336-343).  On power-of-two axes the x-pass
of a migration computes each phase once for both wavefields; on mixed-radix axes, and when one wavefield
marches (modelling, linear adjoint's receiver side), per point.

Bound as in the FP32 tests of the other marches: relative L2 <= 1e-4 against the FP64 oracle, and results that
differ from the FP64-kz ones (the option reaches the kernels).
"""
import numpy as np
import pytest

import oracle as O
import seiswem
from conftest import rel_l2
from test_gpu_parity3d import TOL, oparams_mode, pspi3d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("nx,ny,nz", [(64, 64, 8), (128, 64, 6), (256, 64, 4), (50, 40, 8)])
def test_fp32_pspi(gpu, nx, ny, nz, mode):
    g, vel, refl, wav, sx, sy = pspi3d(nx, ny, nz)
    d = np.random.default_rng(nx + ny + nz).standard_normal((g.nm, g.nt)).astype(np.float32)
    p = oparams_mode(g, mode)
    kw = dict(vel=vel, wav=wav, geom=g, sx=sx, sy=sy, pspi_mode=mode)
    mig = seiswem.ShotProfileWEM(d[None], True, precision=seiswem.PREC_FP32, **kw)
    mod = seiswem.ShotProfileWEM(refl, False, precision=seiswem.PREC_FP32, **kw)[0]
    e1 = rel_l2(mig, O.wem(p, vel, wav, float(sx[0]), float(sy[0]), d=d, adj=True))
    e2 = rel_l2(mod, O.wem(p, vel, wav, float(sx[0]), float(sy[0]), m=refl, adj=False))
    print(f"{nx}x{ny}x{nz} mode={mode}: migrate {e1:.3e} model {e2:.3e}", flush=True)
    assert e1 <= TOL and e2 <= TOL
    assert not np.array_equal(mig, seiswem.ShotProfileWEM(d[None], True, **kw))
