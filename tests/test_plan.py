"""Host arithmetic of the kernels and their launches (csrc/puff_plan.hpp),
compiled alone with the host compiler: no GPU needed."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "puffin_amd", "csrc")

SOURCE = r"""
#include "puff_plan.hpp"
using namespace puff;
extern "C" uint32_t component(int node, int part) { return node_component(node, part); }
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
    return lib


@pytest.mark.parametrize("node", [0, 1, 2 ** 30 - 1, 2 ** 30, 2 ** 31 - 2])
@pytest.mark.parametrize("part", [0, 1])
def test_components_of_the_largest_meshes(plan, node, part):
    """Every mesh that a context admits: below 2^31 nodes."""
    assert plan.component(node, part) == 2 * node + part
