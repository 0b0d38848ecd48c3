"""Mixed precision: the FP32 trailing updates sum no more products than the
shortest panels do unless the caller asks for wider ones.  Shown by a solve that
stops after its first correction, whose error is that of the factor."""
import numpy as np
import pytest

from fedempy_amd import gpu, parts

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def problem():
    p = parts.hex_block(30, 22, 20, 0.3, 0.22, 0.2, seed=3, n_ext=6)
    R = gpu.GpuReducer()
    R.set_part(p)
    z = R.analyze()
    R.reduce()
    F = np.random.default_rng(1).normal(size=(z["ndof1"], 12))
    X = R.solve_internal(F)
    R.close()
    return p, F, X


def first_correction(problem, **options):
    p, F, X = problem
    R = gpu.GpuReducer()
    for k, v in dict(mixedPrecision=1, refineTol=1e30, **options).items():
        R.set_option(k, v)
    R.set_part(p)
    R.analyze()
    R.reduce()
    Y = R.solve_internal(F)
    R.close()
    return np.linalg.norm(Y - X) / np.linalg.norm(X)


def test_default_panels_are_the_shortest(problem):
    short, wide, default = (first_correction(problem, **o) for o in ({"factorPanel": 64}, {"factorPanel": 256}, {}))
    print("64: %.2e  256: %.2e  default: %.2e" % (short, wide, default), flush=True)
    # sums of a quarter of the length are at least as good on this block
    assert short < wide
    assert default <= 1.05 * short
