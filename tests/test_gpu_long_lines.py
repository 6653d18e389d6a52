"""x lines whose plan does not fit a workgroup's LDS are refused before anything
is launched; lengths next to them run."""
import numpy as np
import pytest

from puffin_amd import gpu
from puffin_amd.params import FP64, MIXED, ModuleParams

pytestmark = pytest.mark.gpu


def _mp(nx):
    return ModuleParams(nx=nx, ny=2, nz2=3, dx=0.3, dy=0.3, dz2=0.01, rho=0.01, eta=1e-4, kappa=0.5, gamma_r=100.0,
                        aw=1.0, nbx=4, nby=0, nbz2=0, filt_cutoff=15.0, beta=1.0)


@pytest.mark.parametrize("nx,precision", [(3299, FP64), (6563, MIXED)])
def test_field_stays_where_a_line_does_not_fit(nx, precision):
    print(f"[gpu-lines] refused nx={nx}", flush=True)
    mp = _mp(nx)
    rng = np.random.default_rng(1)
    ar, ai = (rng.standard_normal(mp.nmesh).astype(np.float32).astype(np.float64) for _ in range(2))
    with gpu.Integrator(mp, 1, precision) as g:
        g.upload_field(ar, ai)
        for call in (lambda: g.diffraction_step(0.05), lambda: g.transform(-1)):
            with pytest.raises(gpu.PuffinError, match="does not fit"):
                call()
        gr, gi = g.download_field()
        g.adjoint_enable()
        g.adjoint_upload(None, ar, ai)
        with pytest.raises(gpu.PuffinError, match="does not fit"):
            g.diffraction_adjoint(0.05)
        _, lr, li = g.adjoint_download()
    for got, want in ((gr, ar), (gi, ai), (lr, ar), (li, ai)):
        assert np.array_equal(got, want)


@pytest.mark.parametrize("nx,precision", [(3277, FP64), (3328, FP64), (6553, MIXED), (6554, MIXED)])
def test_lengths_next_to_them_match_numpy(nx, precision):
    """The longest lines in two buffers, and 16 x 16 x 13 in one; 1e-13 and 2e-6 of the largest
    value as for the other lengths, times sqrt(nx / 256) for the direct sums."""
    print(f"[gpu-lines] nx={nx}", flush=True)
    mp = _mp(nx)
    rng = np.random.default_rng(2)
    a = rng.standard_normal((3, 2, nx)) + 1j * rng.standard_normal((3, 2, nx))
    with gpu.Integrator(mp, 1, precision) as g:
        g.upload_field(a.real.reshape(-1).copy(), a.imag.reshape(-1).copy())
        g.transform(-1)
        ar, ai = g.download_field()
    want = np.fft.fftn(a)
    tol = (1e-13 if precision == FP64 else 2e-6) * np.sqrt(nx / 256)
    assert np.abs((ar + 1j * ai).reshape(a.shape) - want).max() / np.abs(want).max() < tol
