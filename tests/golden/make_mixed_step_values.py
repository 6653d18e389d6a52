"""Writes mixed_step_values.npz: p_x, p_y and z2 of a few macroparticles after
seven mixed-form steps in each kind of undulator, by the library given (the
values held are of the stage kernels before their sums were written as FMAs).

    python tests/golden/make_mixed_step_values.py path/to/libpuffin_gpu.so"""
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path[:0] = [ROOT, os.path.join(ROOT, "oracle"), os.path.join(ROOT, "tests")]

if __name__ == "__main__":
    from puffin_amd import gpu
    gpu.LIB_PATH = sys.argv[1]
    from test_gpu_mixed_roundings import CASES, run
    out = {f"{name}_{k}": v for name in CASES for k, v in run(name).items()}
    np.savez(os.path.join(sys.argv[2] if len(sys.argv) > 2 else os.path.dirname(os.path.abspath(__file__)),
                          "mixed_step_values.npz"), **out)
