"""Host arithmetic of the kernels and their launches (csrc/puff_plan.hpp),
compiled alone with the host compiler: no GPU needed."""
import ctypes
import os
import subprocess
import time

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "puffin_amd", "csrc")

SOURCE = r"""
#include <random>
#include <vector>
#include "puff_plan.hpp"
using namespace puff;
template <typename R>
static double sincos_error(double lo, double hi, int n) {
    std::mt19937_64 g(1);
    std::uniform_real_distribution<double> u(std::log(lo), std::log(hi));
    long double worst = 0;
    for (int i = 0; i < n; ++i) {
        const double th = (i & 1 ? -1 : 1) * std::exp(u(g));
        const SinCos<R> t = sincos_phase<R>(th);
        worst = std::max({worst, std::fabs((long double)t.s - sinl(th)), std::fabs((long double)t.c - cosl(th))});
    }
    return (double)worst;
}
extern "C" double sincos_error(int form, double lo, double hi, int n) {
    return form ? sincos_error<float>(lo, hi, n) : sincos_error<double>(lo, hi, n);
}
struct Axis { int n, npass, radix[16], rader; };
static Axis axis_of(int n) {
    Axis a{};
    const bool rader = rader_line(n);
    factorize(rader ? n - 1 : n, a);
    a.n = n;
    a.rader = rader;
    return a;
}
extern "C" void line(int n, int elem, int axis, int cols, int rows, long long* out) {   // B, kind, LDS, fits, radices
    const Axis a = axis_of(n);
    const LinePlan lp = axis_plan(a, elem, axis, cols, rows);
    const long long v[] = {lp.B, lp.kind, (long long)line_lds(a, lp.B, lp.kind, elem, axis), line_fits(a, elem, axis)};
    for (int k = 0; k < 4; ++k) out[k] = v[k];
    for (int k = 0; k < 16; ++k) out[4 + k] = k < a.npass ? a.radix[k] : 0;
}
extern "C" uint32_t component(int node, int part) { return node_component(node, part); }
extern "C" double phase_rate(const double* x, const double* y, const double* z, int nx, int ny, int nz) {
    return largest_phase_rate(std::vector<double>(x, x + nx), std::vector<double>(y, y + ny), std::vector<double>(z, z + nz));
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src, so = d / "plan.cpp", d / "plan.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(so)],
                   check=True)
    lib = ctypes.CDLL(str(so))
    lib.component.restype = ctypes.c_uint32
    lib.phase_rate.restype = lib.sincos_error.restype = ctypes.c_double
    lib.sincos_error.argtypes = [ctypes.c_int, ctypes.c_double, ctypes.c_double, ctypes.c_int]
    return lib


@pytest.mark.parametrize("node", [0, 1, 2 ** 30 - 1, 2 ** 30, 2 ** 31 - 2])
@pytest.mark.parametrize("part", [0, 1])
def test_components_of_the_largest_meshes(plan, node, part):
    """Every mesh that a context admits: below 2^31 nodes."""
    assert plan.component(node, part) == 2 * node + part


def _phase_rate(plan, *k):
    k = [np.ascontiguousarray(v, dtype=np.float64) for v in k]
    dp = ctypes.POINTER(ctypes.c_double)
    return plan.phase_rate(*[v.ctypes.data_as(dp) for v in k], *[v.size for v in k])


def test_phase_rate_is_the_largest_of_all_wavenumbers(plan):
    rng = np.random.default_rng(3)
    kx, ky, kz = rng.standard_normal(7), rng.standard_normal(9), rng.standard_normal(11)
    kz[4] = 0.0
    want = max((x * x + y * y) / abs(2 * z) for x in kx for y in ky for z in kz if z)
    assert abs(_phase_rate(plan, kx, ky, kz) - want) <= 4e-16 * want
    assert _phase_rate(plan, kx, ky, np.zeros(3)) == 0.0


def test_phase_rate_takes_one_pass_over_each_axis(plan):
    """2 10^5 wavenumbers a side: 6 10^5 steps are milliseconds; an axis walked
    again for every wavenumber of another is 8 10^10 of them, most of a minute."""
    k = np.linspace(-1.0, 1.0, 200001)
    t = time.perf_counter()
    _phase_rate(plan, k, k, k)
    assert time.perf_counter() - t < 5.0


@pytest.mark.parametrize("cols,rows", [(10 ** 6, 1000), (26, 26), (1, 1)])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("elem", [16, 8])
def test_plans_of_every_admitted_line(plan, elem, axis, cols, rows):
    """Lengths of 3 n elements within a CU's 160 KiB of LDS: the plan fits too or
    is refused, which only x lines within 4 % of the limit are; the butterflies
    of passes in place fit the registers and the prime pass's tiles the
    accumulators; few lines spread over the chip, but never over part-filled
    tiles where there could be whole ones."""
    out, most = (ctypes.c_longlong * 20)(), (ctypes.c_longlong * 20)()
    for n in range(2, 160 * 1024 // (3 * elem) + 1):
        plan.line(n, elem, axis, cols, rows, out)
        plan.line(n, elem, axis, 10 ** 6, 1000, most)
        B, kind, lds, fits = out[:4]
        radix = [r for r in out[4:] if r]
        assert 1 <= B <= most[0] and kind == most[1], n
        assert (lds <= 160 * 1024) == bool(fits), n
        assert fits or (axis == 0 and 3 * n * elem > 0.96 * 160 * 1024), n
        if kind != 2 and -(-cols // B) * rows < 192:
            assert B // 2 < (min(most[0], -(-8 * radix[0] // n)) if kind == 1 else 1), n
        if n != 257:
            assert np.prod(radix) == n, n
        for k, r in enumerate(radix):
            if kind == 0 or (kind == 1 and k > 0):
                assert r <= 16 and B * (n // r) <= (16 // r) * 256, n
            elif kind == 1:
                assert -(-B * (n // r) // 8) * (((r - 1) // 2 + 16) // 16) <= 16, n


@pytest.mark.parametrize("form,bound", [(0, 9.5e-17), (1, 7.5e-8)])
@pytest.mark.parametrize("decade", [-6, -1, 0, 1, 3, 5, 8, 10, 12])
def test_sine_and_cosine_of_phases(plan, decade, form, bound):
    """The stated bounds against the long double functions (64-bit significand),
    at phases of either sign up to the limit of 1e13."""
    assert plan.sincos_error(form, 10.0 ** decade, 10.0 ** (decade + 1), 200000) < bound
