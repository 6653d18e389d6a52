"""Binned sums over stretches of slots long enough for runs (more than one turn of
a wavefront for the slice sums and the bunching, more than eight for the current):
sorted slots, slots in no order, and stretches that start in order and lose it."""
import math

import numpy as np
import pytest

import oracle as orc
from puffin_amd import gpu
from puffin_amd.params import FP64, MIXED, PI_REF
from test_gpu_macroparticles import _case, _rel

pytestmark = pytest.mark.gpu

SUMS = ("sdata", "aveX", "aveY", "avePX", "avePY", "aveGamma")


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("order", ["sorted", "none", "partly"])
@pytest.mark.parametrize("n", [262145, 600011, 2097217])
def test_sums_of_long_stretches_match_oracle(n, order, precision):
    """1e-10 as for the shorter ones; the mixed form's x, y, p and charge are the
    oracle's rounded to FP32 first, the same values."""
    print(f"[gpu-runs] n={n} {order} precision={precision}", flush=True)
    mp, p, _ = _case(n)
    if order == "partly":   # in the order of z2 but for every seventh
        z = np.sort(p["z2"])
        z[::7] = p["z2"][::7]
        p["z2"] = z
    if precision == MIXED:
        for k in ("x", "y", "px", "py", "chi"):
            p[k] = p[k].astype(np.float32).astype(np.float64)
    zero = np.zeros(mp.nmesh)
    o = orc.Oracle(mp, p, (zero, zero))
    L = 4.0 * PI_REF * mp.rho
    ns = int(math.ceil(mp.nz2 * mp.dz2 / L)) + 1
    with gpu.Integrator(mp, n, precision) as g:
        g.upload_particles(p)
        if order == "sorted":
            g.sort_now()
        st, want = o.slice_stats(ns, L)
        got = g.slice_stats(ns, L)
        assert st == 0
        for k in SUMS:
            assert _rel(got[k], want[k], 1.0) < 1e-10, k
        assert _rel(g.bunching(1, ns, L), o.bunching(1, ns, L)) < 1e-10
        st, cur = o.current(mp.nz2 + 1, mp.dz2)
        assert st == 0 and _rel(g.current(mp.nz2 + 1, mp.dz2), cur) < 1e-10
