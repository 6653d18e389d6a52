"""Kernels over macroparticles at the counts and beams where they can go
wrong: one macroparticle, partial wavefronts and workgroups, sorted beams so
thin that a workgroup's cells do not fit its LDS tile (its wavefronts deposit
in turn, or straight to memory), and odd counts through the records of the
sort, the uploads and the downloads.

Tolerances: FP64 1e-10 of the largest value, as for the other runs against the
oracle; the mixed form 1e-5 (x, y, p and the field are FP32, and a deposit is
rounded to 2^-22 of its workgroup's largest), z2 and Gamma 1e-8."""
import math

import numpy as np
import pytest

import oracle as orc
from puffin_amd import gpu
from puffin_amd.configs import match_in
from puffin_amd.params import FP64, MIXED, PI_REF, UND_ELLIPTICAL, UND_PLANEPOLE, ModuleParams, scaling, step_size

pytestmark = pytest.mark.gpu

KEYS = ("x", "y", "z2", "px", "py", "gam")


def _rel(got, want, least=1e-300):
    return float(np.abs(np.asarray(got) - want).max() / max(np.abs(want).max(), least))


def _case(n, und_type=UND_ELLIPTICAL, nx=33, nz2=200):
    rho = 0.01
    eta, kappa, fx, fy = scaling(rho, 1.0, 100.0, 1 / math.sqrt(2), 1 / math.sqrt(2))
    h = step_size(rho, 30)
    mp = ModuleParams(nx=nx, ny=nx, nz2=nz2, dx=0.2, dy=0.2, dz2=4 * PI_REF * rho / 16, rho=rho, eta=eta, kappa=kappa,
                      gamma_r=100.0, aw=1.0, fx=fx, fy=fy, und_type=und_type, szfs=0.0, szfe=60 * h, nbx=4, nby=4,
                      nbz2=9, filt_cutoff=10.0)
    rng = np.random.default_rng(n)
    lz = (nz2 - 1) * mp.dz2
    p = dict(x=np.clip(rng.standard_normal(n), -2.5, 2.5), y=np.clip(rng.standard_normal(n), -2.5, 2.5),
             z2=rng.uniform(0.05, 0.6 * lz, n), px=np.zeros(n), py=np.zeros(n),
             gam=1.0 + 1e-3 * rng.standard_normal(n), chi=np.full(n, 2 * math.pi * lz / n))
    match_in(mp, 1.0, p)
    return mp, p, h


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("und_type", [UND_ELLIPTICAL, UND_PLANEPOLE])
@pytest.mark.parametrize("n", [1, 63, 257, 1025, 20011])
def test_thin_sorted_beams_match_oracle(n, und_type, precision):
    print(f"[gpu-particles] stages n={n} und={und_type} precision={precision}", flush=True)
    mp, p, h = _case(n, und_type)
    zero = np.zeros(mp.nmesh)
    o = orc.Oracle(mp, p, (zero.copy(), zero.copy()), taper=(1.0, 1.0, -0.01))
    with gpu.Integrator(mp, n, precision) as g:
        g.upload_particles(p)
        g.upload_field(zero, zero)
        g.set_taper(1.0, 1.0, -0.01)
        g.sort_now()
        szl = 0.0
        for _ in range(3):
            assert o.rk4par(szl, h) == 0
            assert g.rk4par(szl, h) == 0
            szl += h
        out = g.download_particles()
        gr, gi = g.download_field()
    for k in KEYS:
        tol = 1e-10 if precision == FP64 else (1e-8 if k in ("z2", "gam") else 1e-5)
        assert _rel(out[k], o.parts[k], 1.0 if k in ("px", "py") else 1e-300) < tol, k
    scale = np.abs(o.ar + 1j * o.ai).max()
    assert np.abs((gr - o.ar) + 1j * (gi - o.ai)).max() / scale < (1e-10 if precision == FP64 else 1e-5)


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("n", [1, 2, 255, 257, 100003])
def test_records_keep_every_macroparticle(n, precision):
    """Host and device uploads, a sort, and downloads in the caller's order
    return what was given, rounded to the form's types."""
    import torch
    mp, p, _ = _case(n)
    want = {k: (p[k] if precision == FP64 or k in ("z2", "gam") else p[k].astype(np.float32).astype(np.float64))
            for k in KEYS}
    with gpu.Integrator(mp, n, precision) as g:
        for device in (False, True):
            if device:
                g.upload_particles_torch({k: torch.from_numpy(p[k]).to("cuda") for k in KEYS + ("chi",)})
            else:
                g.upload_particles(p)
            for _ in range(2):
                g.sort_now()
            host = g.download_particles()
            dev = g.download_particles_torch()
            for k in KEYS:
                assert np.array_equal(host[k], want[k]), (k, device)
                assert np.array_equal(dev[k].cpu().numpy(), want[k]), (k, device)


@pytest.mark.parametrize("in_order", [False, True])
@pytest.mark.parametrize("n", [1, 63, 65, 4099, 50001])
def test_diagnostics_match_oracle(n, in_order):
    """Sums per slice from runs of slots in one slice (sorted) and from slots
    in any order.  Widths are roots of differences that round at 1e-16: 1e-7.
    (The beam's momenta are equal: their widths and the emittances are roots
    of rounding alone, and not compared.)"""
    mp, p, _ = _case(n)
    rng = np.random.default_rng(2)
    ar, ai = rng.standard_normal(mp.nmesh), rng.standard_normal(mp.nmesh)
    o = orc.Oracle(mp, p, (ar, ai))
    L = 4.0 * PI_REF * mp.rho
    ns = int(math.ceil(mp.nz2 * mp.dz2 / L)) + 1
    with gpu.Integrator(mp, n, FP64) as g:
        g.upload_particles(p)
        g.upload_field(ar, ai)
        if in_order:
            g.sort_now()
        st, want = o.slice_stats(ns, L)
        got = g.slice_stats(ns, L)
        assert st == 0
        for k in set(want) - {"sdpX", "sdpY", "eX", "eY"}:
            tol = 1e-10 if k in ("sdata", "aveX", "aveY", "avePX", "avePY", "aveGamma") else 1e-7
            assert _rel(got[k], want[k], 1.0) < tol, k
        for hm in (1, 2):
            assert _rel(g.bunching(hm, ns, L), o.bunching(hm, ns, L)) < 1e-10
        st, cur = o.current(mp.nz2 + 1, mp.dz2)
        assert st == 0 and _rel(g.current(mp.nz2 + 1, mp.dz2), cur) < 1e-10
        assert _rel(g.power(), o.power()) < 1e-10


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("n", [1, 63, 65, 257, 100003])
def test_corrector_matches_oracle(n, precision):
    mp, p, _ = _case(n)
    rng = np.random.default_rng(4)
    p["x"], p["px"] = p["x"] + 0.3, p["px"] + 0.1 * rng.standard_normal(n)
    want = {k: p[k].copy() for k in p}
    orc.correct_trans(want)
    with gpu.Integrator(mp, n, precision) as g:
        g.upload_particles(p)
        g.correct_trans()
        out = g.download_particles()
    for k in ("x", "y", "px", "py"):
        assert _rel(out[k], want[k], 1.0) < (1e-12 if precision == FP64 else 1e-6), k
