"""The first load case of a process takes no scratch array of the entry
without allocation (32 MiB, loaded with its code object)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CHILD = """
import ctypes, sys
sys.path.insert(0, sys.argv[1])
import numpy as np
from fedempy_amd import gpu, parts
R = gpu.GpuReducer()
R.set_part(parts.hex_block(7, 5, 4, 0.07, 0.05, 0.04, seed=6, n_ext=5))
z = R.analyze(ngen=2)
R.reduce()
hip = ctypes.CDLL("libamdhip64.so")
def free():
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value
F = np.ones((z["neq"], 1), order="F")
out = np.zeros((z["ndim"], 1), order="F")
before = free()
assert R.lib.fgpu_reduce_loads(R.h, 1, gpu._ptr(F), gpu._ptr(out)) == 0
print("taken", before - free())
"""


def test_first_load_case_takes_no_scratch_array():
    pkg = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fedem-solvers_amd")
    r = subprocess.run([sys.executable, "-c", CHILD, pkg], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    assert int(r.stdout.split()[-1]) < 24 << 20
