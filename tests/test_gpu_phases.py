"""The propagator's rotation at phases of a fraction to 1e13 and past the limit of
the registers' sine and cosine, against numpy: the complex field, z2 lines in
registers and through LDS, either sign of kz and of the step, and the adjoint.

The mesh's lengths make kx and ky whole numbers, so that a phase is rounded once
and is the same double in numpy: the bounds of a diffraction step (1e-12 and
5e-6 of the largest value) hold at every phase."""
import math

import numpy as np
import pytest

from puffin_amd import gpu
from puffin_amd.params import FP64, MIXED, ModuleParams

pytestmark = pytest.mark.gpu

PI = 4.0 * math.atan(1.0)


def _k(n, length):
    i = np.arange(n)
    i[i >= math.ceil(n / 2)] -= n
    return 2.0 * PI * i / length


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("phase", [3.0, -3.0, 1e3, 1e8, 0.9999e13, 1.0001e13, 3e16])
@pytest.mark.parametrize("nz", [128, 512, 4096, 96, 106, 257])
def test_rotation_matches_numpy(nz, phase, precision):
    print(f"[gpu-phases] nz={nz} phase={phase} precision={precision}", flush=True)
    nx, ny = 4, 8
    mp = ModuleParams(nx=nx, ny=ny, nz2=nz, dx=2 * PI / nx, dy=2 * PI / ny, dz2=2 * PI / nz, rho=0.01, eta=1e-4,
                      kappa=0.5, gamma_r=100.0, aw=1.0, nbz2=0, filt_cutoff=0.0, filter=0, beta=0.0)
    kx, ky, kz = _k(nx, nx * mp.dx), _k(ny, ny * mp.dy), _k(nz, nz * mp.dz2)
    assert np.array_equal(kx, np.rint(kx)) and np.array_equal(ky, np.rint(ky))
    k2 = (kx ** 2)[None, None, :] + (ky ** 2)[None, :, None]
    nonzero = kz != 0.0
    h = phase / (k2.max() / np.abs(2 * kz[nonzero]).min())
    h = float(np.float32(h))   # h k2 is exact
    th = np.zeros((nz, ny, nx))
    kzn = kz[nonzero][:, None, None]
    th[nonzero] = h * k2 / (2.0 * kzn) if precision == FP64 else h * k2 * (1.0 / (2.0 * kzn))
    rng = np.random.default_rng(5)
    a = rng.standard_normal((nz, ny, nx)) + 1j * rng.standard_normal((nz, ny, nx))
    fwd = np.fft.ifftn(np.fft.fftn(a) * (np.cos(th) + 1j * np.sin(th)))
    adj = np.fft.ifftn(np.fft.fftn(a) * (np.cos(th) - 1j * np.sin(th)))
    re, im = a.real.reshape(-1).copy(), a.imag.reshape(-1).copy()
    with gpu.Integrator(mp, 1, precision) as g:
        g.upload_field(re, im)
        g.diffraction_step(h)
        gr, gi = g.download_field()
        g.adjoint_enable()
        g.adjoint_upload(None, re, im)
        g.diffraction_adjoint(h)
        _, lr, li = g.adjoint_download()
    tol = 1e-12 if precision == FP64 else 5e-6
    for got, want in ((gr + 1j * gi, fwd), (lr + 1j * li, adj)):
        assert np.abs(got.reshape(a.shape) - want).max() / np.abs(want).max() < tol
