"""Elastic migration and modelling around 2 nmx = nkx on power-of-two lengths, where the two potentials go
through the transforms in lockstep and the zero half of the line is dropped (pad factor 2 and up) or kept
(pad factor 1), with the source below the receivers (single steps beside the lockstep ones).

Bound as at every other size: relative L2 <= 1e-4 against the FP64 oracle.
"""
import numpy as np
import pytest

import oracle as O
from conftest import rel_l2
from test_gpu_ewem import TOL, case, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("below", [0.0, 2.5])
@pytest.mark.parametrize("nx,padx", [(128, 1), (512, 1), (256, 2), (512, 2), (1024, 2), (256, 4)])
def test_ewem_pow2_lengths(gpu, nx, padx, below):
    g, p, vp, vs, wav, rng = case(nx, nz=8, nt=128, seed=nx + padx)
    g.padx = p.padx = padx
    g.sz = p.sz = g.oz + below * g.dz
    sx = g.dmx * (nx // 3)
    ux, uy, uz = rng.standard_normal((3, g.nm, g.nt)).astype(np.float32)
    mpp, _, mps2 = run(g, vp, vs, wav, sx, True, ux, uy, uz)
    rpp, rps2 = O.ewem(p, vp, vs, wav, sx, ux=ux, uz=uz, adj=True)
    m1, m2 = rng.standard_normal((2, g.nm, g.nz)).astype(np.float32)
    dx, _, dz = run(g, vp, vs, wav, sx, False, m1, np.zeros_like(m1), m2)
    rx, rz = O.ewem(p, vp, vs, wav, sx, mpp=m1, mps2=m2, adj=False)
    errs = [rel_l2(mpp, rpp), rel_l2(mps2, rps2), rel_l2(dx, rx), rel_l2(dz, rz)]
    print(f"nkx={nx * padx} below={below}: PP {errs[0]:.3e} PS {errs[1]:.3e} ux {errs[2]:.3e} uz {errs[3]:.3e}", flush=True)
    assert max(errs) <= TOL
