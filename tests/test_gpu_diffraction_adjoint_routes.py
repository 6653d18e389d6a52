"""The diffraction's adjoint on every route of its x, y and z2 lines, in both
forms: 257 points in registers, compiled plans, the matrix pass, one and two
LDS buffers, z2 lines in registers.

Tolerances: 1e-12 of the largest value as for the other adjoints, and the mixed
form's 5e-6 of a diffraction step."""
import numpy as np
import pytest

import oracle as orc
from puffin_amd import gpu
from puffin_amd.params import FP64, MIXED, ModuleParams

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("periodic", [0, 1])
@pytest.mark.parametrize("shape", [(257, 5, 12), (5, 257, 12), (257, 257, 3), (129, 33, 10), (33, 129, 10),
                                   (61, 47, 53), (17, 34, 59), (10, 15, 84), (29 * 23, 5, 7), (5, 4, 512)])
def test_adjoint_matches_oracle(shape, periodic, precision):
    print(f"[gpu-adjoint] shape={shape} periodic={periodic} precision={precision}", flush=True)
    nx, ny, nz = shape
    mp = ModuleParams(nx=nx, ny=ny, nz2=nz + periodic, dx=0.3, dy=0.3, dz2=0.01, rho=0.01, eta=1e-4, kappa=0.5,
                      gamma_r=100.0, aw=1.0, periodic=periodic, nbz2=1, filt_cutoff=15.0, beta=1.0)
    rng = np.random.default_rng(9)
    y = rng.standard_normal(mp.nmesh) + 1j * rng.standard_normal(mp.nmesh)
    lr, li = y.real.copy(), y.imag.copy()
    orc.diffraction_adjoint(mp, lr, li, 0.0837)
    p = dict(x=np.zeros(1), y=np.zeros(1), z2=np.full(1, 0.01), px=np.zeros(1), py=np.zeros(1), gam=np.ones(1),
             chi=np.zeros(1))
    with gpu.Integrator(mp, 1, precision) as g:
        g.upload_particles(p)
        g.adjoint_enable()
        g.adjoint_upload(None, y.real.copy(), y.imag.copy())
        g.diffraction_adjoint(0.0837)
        _, gr, gi = g.adjoint_download()
    want = lr + 1j * li
    tol = 1e-12 if precision == FP64 else 5e-6
    assert np.abs(gr + 1j * gi - want).max() / np.abs(want).max() < tol
