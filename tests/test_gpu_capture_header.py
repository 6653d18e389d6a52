"""A step capture names its layout: one written by a library with another layout
(all six stage derivatives kept) is refused, not read at this one's offsets."""
import numpy as np
import pytest

from puffin_amd import gpu
from puffin_amd.params import FP64, ModuleParams

pytestmark = pytest.mark.gpu


def test_capture_of_another_layout_is_refused():
    import torch
    print("[gpu] capture header", flush=True)
    n = 65
    mp = ModuleParams(nx=9, ny=9, nz2=32, dx=0.5, dy=0.5, dz2=0.01, rho=0.01, eta=1e-4, kappa=0.5, gamma_r=100.0,
                      aw=1.0, szfs=0.0, szfe=1.0, nbx=2, nby=2, nbz2=4, filt_cutoff=10.0)
    rng = np.random.default_rng(1)
    p = dict(x=rng.uniform(-1, 1, n), y=rng.uniform(-1, 1, n), z2=rng.uniform(0.05, 0.2, n), px=np.zeros(n),
             py=np.zeros(n), gam=np.ones(n), chi=np.full(n, 1e-3))
    zero = np.zeros(mp.nmesh)
    with gpu.Integrator(mp, n, FP64) as g:
        g.upload_particles(p)
        g.upload_field(zero, zero)
        g.adjoint_enable()
        g.adjoint_zero()
        cap = torch.empty(g.capture_bytes(), dtype=torch.uint8, device="cuda")
        hdr = np.zeros(gpu.STATE_HEADER_BYTES, dtype=np.uint8)
        assert g.rk4par_capture(0.0, 1e-3, cap.data_ptr(), hdr) == 0
        older = hdr.copy()
        older[:8] = np.frombuffer(b"PUFFCAP1", dtype=np.uint8)
        with pytest.raises(gpu.PuffinError, match="capture"):
            g.rk4par_adjoint_captured(0.0, 1e-3, cap.data_ptr(), older)
        st, _, _ = g.rk4par_adjoint_captured(0.0, 1e-3, cap.data_ptr(), hdr)
        assert st == 0
