"""Line transforms of every pass and route against numpy and the oracle: the
passes of 2 to 16 points alone and combined, in one and in two LDS buffers,
direct passes of larger primes, and z2 lines of a power of two in registers
(odd and even numbers of columns, a last workgroup that is partly empty).

Tolerances as for the other transforms: 1e-13 and 2e-6 of the largest value
(a few rounding errors per pass), 1e-12 and 5e-6 for a diffraction step (six
transforms and the spectral factors)."""
import numpy as np
import pytest

import oracle as orc
from puffin_amd import gpu
from puffin_amd.params import FP64, MIXED, ModuleParams

pytestmark = pytest.mark.gpu


def _mp(nx, ny, nz2, **kw):
    return ModuleParams(nx=nx, ny=ny, nz2=nz2, dx=0.3, dy=0.3, dz2=0.01, rho=0.01, eta=1e-4, kappa=0.5,
                        gamma_r=100.0, aw=1.0, **kw)


def _rel(got, want):
    return np.abs(got - want).max() / np.abs(want).max()


SHAPES = [(r, r, r) for r in range(3, 17)]
SHAPES += [(90, 75, 420),       # 10 9, 15 5, 10 7 6
           (132, 143, 12),      # 12 11, 13 11
           (3, 2, 3388),        # 11 11 7 4: too long for one thread per butterfly
           (61, 47, 34),        # direct passes only; 17 2
           (2, 3, 389),
           (9, 225, 512), (3, 3, 128), (7, 5, 256), (2, 2, 2048), (23, 3, 1024)]


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("shape", SHAPES)
def test_lines_match_numpy(shape, precision):
    nx, ny, nz = shape
    print(f"[gpu-lines] shape={shape} precision={precision}", flush=True)
    mp = _mp(nx, ny, nz)
    rng = np.random.default_rng(7)
    a = rng.standard_normal((nz, ny, nx)) + 1j * rng.standard_normal((nz, ny, nx))
    with gpu.Integrator(mp, 1, precision) as g:
        g.upload_field(a.real.reshape(-1).copy(), a.imag.reshape(-1).copy())
        g.transform(-1)
        ar, ai = g.download_field()
        g.transform(+1)
        br, bi = g.download_field()
    tol = 1e-13 if precision == FP64 else 2e-6
    assert _rel((ar + 1j * ai).reshape(nz, ny, nx), np.fft.fftn(a)) < tol
    assert _rel((br + 1j * bi).reshape(nz, ny, nx), a * (nx * ny * nz)) < tol


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("shape", [(5, 3, 128), (4, 5, 256), (3, 3, 512), (7, 5, 1024), (3, 2, 2048), (13, 9, 2048),
                                   (10, 15, 84), (11, 13, 90)])
def test_diffraction_step_matches_oracle(shape, precision):
    print(f"[gpu-lines] diffraction {shape} precision={precision}", flush=True)
    mp = _mp(*shape, nbz2=9, filt_cutoff=15.0, beta=1.0)
    rng = np.random.default_rng(11)
    ar, ai = rng.standard_normal(mp.nmesh), rng.standard_normal(mp.nmesh)
    zero = np.zeros(1)
    o = orc.Oracle(mp, dict(x=zero, y=zero, z2=zero, px=zero, py=zero, gam=np.ones(1), chi=zero), (ar, ai))
    o.diffraction_step(0.0837)
    with gpu.Integrator(mp, 1, precision) as g:
        g.upload_field(ar, ai)
        g.diffraction_step(0.0837)
        gr, gi = g.download_field()
    tol = 1e-12 if precision == FP64 else 5e-6
    assert _rel(gr + 1j * gi, o.ar + 1j * o.ai) < tol


@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_phases_beyond_the_reduction(precision):
    """Propagator phases past the limit of the registers' sine and cosine take
    the general pass: without a mask or filter the step is a rotation of each
    wavenumber, so the sum of |A|^2 stays (rounding of 2 x 3 transforms)."""
    mp = _mp(4, 6, 128, nbz2=0, filt_cutoff=0.0, filter=0, beta=0.0)
    rng = np.random.default_rng(3)
    ar, ai = rng.standard_normal(mp.nmesh), rng.standard_normal(mp.nmesh)
    with gpu.Integrator(mp, 1, precision) as g:
        g.upload_field(ar, ai)
        g.diffraction_step(1e15)
        gr, gi = g.download_field()
    want = np.sum(ar ** 2 + ai ** 2)
    assert abs(np.sum(gr ** 2 + gi ** 2) - want) / want < (1e-12 if precision == FP64 else 5e-6)
