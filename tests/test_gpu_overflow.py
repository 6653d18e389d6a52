"""Stage workgroups whose node box overflows the LDS tile: sorted beams so thin
that 256 consecutive slots spread over the whole cross-section."""
import math

import numpy as np
import pytest

import oracle as orc
from puffin_amd import gpu
from puffin_amd.configs import match_in
from puffin_amd.params import FP64, MIXED, PI_REF, ModuleParams, scaling, step_size

pytestmark = pytest.mark.gpu


def _beam(n, seed=5):
    rho = 0.01
    eta, kappa, fx, fy = scaling(rho, 1.0, 100.0, 1 / math.sqrt(2), 1 / math.sqrt(2))
    h = step_size(rho, 30)
    mp = ModuleParams(nx=33, ny=33, nz2=200, dx=0.2, dy=0.2, dz2=4 * PI_REF * rho / 16, rho=rho, eta=eta, kappa=kappa,
                      gamma_r=100.0, aw=1.0, fx=fx, fy=fy, szfs=0.0, szfe=60 * h, nbx=4, nby=4, nbz2=9,
                      filt_cutoff=10.0)
    rng = np.random.default_rng(seed)
    lz = (mp.nz2 - 1) * mp.dz2
    p = dict(x=rng.uniform(0.3, 2.7, n) * np.where(rng.random(n) < 0.5, -1.0, 1.0), y=rng.uniform(-2.7, 2.7, n),
             z2=rng.uniform(0.05, 0.6 * lz, n), px=np.zeros(n), py=np.zeros(n),
             gam=1.0 + 1e-3 * rng.standard_normal(n), chi=np.full(n, 2 * math.pi * lz / n))
    match_in(mp, 1.0, p)
    return mp, p, h


@pytest.mark.parametrize("n", [1536, 2048, 3072, 4096, 6144])
def test_light_macroparticles_beside_heavy_ones(n):
    """The mixed form's field of macroparticles 1e-7 as heavy as others of their
    workgroup, on nodes that only they touch (x > 0; the heavy ones stay 0.2, one
    cell, below): FP32 rounding of their own, 1e-5 of their largest as elsewhere
    in this form."""
    mp, p, h = _beam(n)
    p["chi"] = p["chi"] * np.where(p["x"] > 0, 1e-7, 1.0)
    zero = np.zeros(mp.nmesh)
    o = orc.Oracle(mp, p, (zero.copy(), zero.copy()))
    assert o.rk4par(0.0, h) == 0
    with gpu.Integrator(mp, n, MIXED) as g:
        g.upload_particles(p)
        g.upload_field(zero, zero)
        g.sort_now()
        assert g.rk4par(0.0, h) == 0
        share = g.tile_fallback()
        gr, gi = g.download_field()
    print(f"[gpu-overflow] n={n} share={share}", flush=True)
    assert share[-1] == 1.0   # whole workgroups, all overflowing: none takes the packed tile
    shape = (mp.nz2, mp.ny, mp.nx)
    light = np.s_[:, :, mp.nx // 2 + 1:]
    got, want = ((r + 1j * i).reshape(shape)[light] for r, i in ((gr, gi), (o.ar, o.ai)))
    assert np.abs(want).max() > 0
    assert np.abs(got - want).max() / np.abs(want).max() < 1e-5


@pytest.mark.parametrize("n", [63, 2048, 4099])
def test_deterministic_deposit_of_thin_sorted_beams(n):
    """Wavefront by wavefront in fixed point: the bits of the unsorted slots (whose
    wavefronts deposit straight to memory), and the oracle's values to 1e-10."""
    mp, p, h = _beam(n)
    zero = np.zeros(mp.nmesh)
    o = orc.Oracle(mp, p, (zero.copy(), zero.copy()))
    out = []
    for in_order in (False, True):
        print(f"[gpu-overflow] deterministic n={n} sorted={in_order}", flush=True)
        with gpu.Integrator(mp, n, FP64) as g:
            g.set_deterministic(True)
            g.set_sort_interval(0)
            g.upload_particles(p)
            g.upload_field(zero, zero)
            if in_order:
                g.sort_now()
            for k in range(3):
                assert g.rk4par(k * h, h) == 0
            out.append((g.download_particles(), g.download_field()))
    for k in range(3):
        assert o.rk4par(k * h, h) == 0
    for k in ("x", "y", "z2", "px", "py", "gam"):
        assert np.array_equal(out[0][0][k], out[1][0][k]), k
        assert np.abs(out[1][0][k] - o.parts[k]).max() <= 1e-10 * np.abs(o.parts[k]).max(), k
    for a, b in zip(out[0][1], out[1][1]):
        assert np.array_equal(a, b)
    want = o.ar + 1j * o.ai
    assert np.abs(out[1][1][0] + 1j * out[1][1][1] - want).max() <= 1e-10 * np.abs(want).max()
