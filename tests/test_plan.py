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
#include <vector>
#include "puff_plan.hpp"
using namespace puff;
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
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(so)],
                   check=True)
    lib = ctypes.CDLL(str(so))
    lib.component.restype = ctypes.c_uint32
    lib.phase_rate.restype = ctypes.c_double
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
