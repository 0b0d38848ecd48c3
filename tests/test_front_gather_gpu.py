"""Fronts gathered from their children over the sizes where the gather changes
its form: fronts below 16 rows, past 256, 512 and 1024 rows, boundary fronts
of several column blocks, and memory that still holds an earlier factor."""
import numpy as np
import pytest
import scipy.sparse as sp

from fedempy_amd import gpu, parts

pytestmark = pytest.mark.gpu

# a factorisation and two triangular passes: n eps with room for the explicit
# inverses of the pivot blocks (FP64), the refinement's own limit (mixed)
TOL = {False: 1e-12, True: 1e-11}


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("dims,n_ext", [((2, 1, 1), 4), ((5, 4, 3), 3), ((9, 8, 7), 40), ((14, 13, 12), 5), ((17, 16, 15), 9)])
def test_block(dims, n_ext, mixed):
    print("block of", dims, "external nodes", n_ext, "mixed" if mixed else "fp64", flush=True)
    R = gpu.GpuReducer()
    if mixed:
        R.set_option("mixedPrecision", 1)
    R.set_part(parts.hex_block(*dims, *(0.01 * d for d in dims), seed=2, n_ext=n_ext))
    z = R.analyze()
    out = []
    for _ in range(2):  # the second factor starts from the first one's memory
        R.reduce()
        out.append((R.reduced()[0], R.B()))
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    SK, B = out[0]
    rp, ci, K, _, pe = R.csr()
    K = sp.csr_matrix((K, ci, rp), shape=(z["neq"],) * 2)
    n1, eq = z["ndof1"], np.argsort(pe)
    K = K[eq][:, eq]
    X = R.solve_internal(K[:n1, n1:].toarray())
    scale = abs(K).max() * max(1.0, abs(B).max())
    for b in (B, -X):
        assert abs(K[:n1, :n1] @ b + K[:n1, n1:]).max() <= TOL[mixed] * scale
        assert abs(SK - (K[n1:, n1:] + K[n1:, :n1] @ b)).max() <= TOL[mixed] * scale
    R.close()
