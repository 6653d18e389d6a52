"""Lines per workgroup as the mesh gives them: few lines (fewer a workgroup, so
that more of the chip works), many, whole and part-filled tiles of the matrix
pass, its rotations apart by powers of two in the table.

Tolerances as for the other transforms: 1e-13 and 2e-6 of the largest value."""
import numpy as np
import pytest

from puffin_amd import gpu
from puffin_amd.params import FP64, MIXED, ModuleParams

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("shape", [(26, 26, 236), (70, 64, 236),     # 59 4
                                   (26, 24, 934), (3, 2, 1011),      # 467 2, 337 3
                                   (52, 60, 272), (272, 3, 4), (3, 272, 4),   # 17 16
                                   (5, 70, 1684), (389, 30, 3), (30, 389, 3),
                                   (26, 26, 260), (90, 80, 260), (260, 5, 3), (5, 260, 3),
                                   (26, 26, 667), (26, 26, 521)])    # two buffers: 29 23, 521
def test_lines_match_numpy(shape, precision):
    nx, ny, nz = shape
    print(f"[gpu-fill] shape={shape} precision={precision}", flush=True)
    mp = ModuleParams(nx=nx, ny=ny, nz2=nz, dx=0.3, dy=0.3, dz2=0.01, rho=0.01, eta=1e-4, kappa=0.5, gamma_r=100.0,
                      aw=1.0)
    rng = np.random.default_rng(7)
    a = rng.standard_normal((nz, ny, nx)) + 1j * rng.standard_normal((nz, ny, nx))
    with gpu.Integrator(mp, 1, precision) as g:
        g.upload_field(a.real.reshape(-1).copy(), a.imag.reshape(-1).copy())
        g.transform(-1)
        ar, ai = g.download_field()
        g.transform(+1)
        br, bi = g.download_field()
    tol = 1e-13 if precision == FP64 else 2e-6
    f = np.fft.fftn(a)
    assert np.abs((ar + 1j * ai).reshape(a.shape) - f).max() / np.abs(f).max() < tol
    b = a * (nx * ny * nz)
    assert np.abs((br + 1j * bi).reshape(a.shape) - b).max() / np.abs(b).max() < tol
