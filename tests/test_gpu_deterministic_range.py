"""A source that outgrows the deterministic deposit's range within a step is an
error that leaves the state as it was, whichever stage forms it."""
import math

import numpy as np
import pytest

from puffin_amd import gpu
from puffin_amd.params import FP64, PI_REF, ModuleParams, scaling

pytestmark = pytest.mark.gpu

KEYS = ("x", "y", "z2", "px", "py", "gam")


def _case(n, chi):
    rho = 0.01
    eta, kappa, fx, fy = scaling(rho, 1.0, 100.0, 1 / math.sqrt(2), 1 / math.sqrt(2))
    mp = ModuleParams(nx=17, ny=17, nz2=64, dx=0.4, dy=0.4, dz2=4 * PI_REF * rho / 16, rho=rho, eta=eta, kappa=kappa,
                      gamma_r=100.0, aw=1.0, fx=fx, fy=fy, szfs=0.0, szfe=1.0, nbx=4, nby=4, nbz2=9, filt_cutoff=10.0)
    rng = np.random.default_rng(n)
    p = dict(x=rng.uniform(-2, 2, n), y=rng.uniform(-2, 2, n), z2=rng.uniform(0.05, 0.2, n), px=np.zeros(n),
             py=np.zeros(n), gam=np.ones(n), chi=np.full(n, chi))
    return mp, p


def _step(mp, p, h, det):
    zero = np.zeros(mp.nmesh)
    with gpu.Integrator(mp, p["x"].size, FP64) as g:
        g.upload_particles(p)
        g.upload_field(zero, zero)
        g.set_deterministic(det)
        status = 0
        try:
            status = g.rk4par(0.0, h)
        except gpu.PuffinError as e:
            status = e.status
        return status, g.download_particles(), g.download_field()


@pytest.mark.parametrize("n", [1, 65, 200])
def test_source_out_of_range_in_the_last_stage(n):
    """The undulator moves p_x or p_y by d in a step, from d / 4: the sources of the
    four stages are d / 4 times 1, 3, 3 and 5 (the field's phase turns by 0.06).
    The limit lies at 4 / f times the first, f in [1/2, 1) the fraction of
    4 n |s| as a binary number, here 0.9: only stage 4 exceeds it.  As many
    macroparticles as one workgroup holds at most."""
    print(f"[gpu-det] range n={n}", flush=True)
    h = 1.1e-3
    mp, p = _case(n, 1e-3)
    _, q, _ = _step(mp, p, h, False)
    k = max(("px", "py"), key=lambda k: abs(q[k][0]))
    start = q[k][0] / 4
    gamma_z = 1.0 / math.sqrt(1.0 - (1.0 + start ** 2) / mp.gamma_r ** 2)
    s = abs(start) * gamma_z / (mp.dx * mp.dy * mp.dz2)
    chi = 0.9 * 2.0 ** -20 / (4 * n * s)
    mp, p = _case(n, chi)
    p[k] += start
    status, q, (ar, ai) = _step(mp, p, h, True)
    assert status not in (0, 1, 2, 3)
    for j in KEYS:
        assert np.array_equal(q[j], p[j]), j
    assert not ar.any() and not ai.any()
    # the same step is in range with a start ten times as large
    p[k] *= 10
    status, q, (ar, ai) = _step(mp, p, h, True)
    assert status == 0 and not np.array_equal(q[k], p[k]) and ar.any()
