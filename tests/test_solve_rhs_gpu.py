"""Solves with the resident factor over the right-hand side counts where the
products change their form (16-column tiles, groups of up to 96 columns) and
over fused and unfused levels."""
import numpy as np
import pytest
import scipy.sparse as sp

from fedempy_amd import gpu, parts

pytestmark = pytest.mark.gpu


def solver(part, mixed=False, **kw):
    R = gpu.GpuReducer()
    if mixed:
        R.set_option("mixedPrecision", 1)
    R.set_part(part)
    z = R.analyze(**kw)
    R.reduce()
    rp, ci, K, _, pe = R.csr()
    A = sp.csr_matrix((K, ci, rp), shape=(z["neq"],) * 2)
    eq = np.argsort(pe)[:z["ndof1"]]  # permuted row of every internal equation
    return R, A[eq][:, eq], z["ndof1"]


def backward_error(A, X, F):
    """largest column's |F - A X| over |A| |X| + |F| (norms)"""
    a = np.sqrt((A.multiply(A)).sum())
    r = np.linalg.norm(F - A @ X, axis=0)
    return float(np.max(r / (a * np.linalg.norm(X, axis=0) + np.linalg.norm(F, axis=0))))


# a factorisation and two triangular passes of n equations: n eps with room
# for the explicit inverses of the pivot blocks
TOL = 1e-12


@pytest.fixture(scope="module")
def plate():
    p = parts.plate(21, 17, 0.42, 0.34, ext_nodes=[0, 17, 378, 395])
    s = {m: solver(p, mixed=m) for m in (False, True)}
    yield s
    for R, _, _ in s.values():
        R.close()


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("nrhs", [1, 3, 15, 16, 17, 24, 33, 64, 80, 95, 96, 97, 193])
def test_right_hand_side_counts(plate, nrhs, mixed):
    print("nrhs", nrhs, "mixed" if mixed else "fp64", flush=True)
    R, A, n1 = plate[mixed]
    F = np.random.default_rng(nrhs).normal(0.0, 1.0, (n1, nrhs))
    X = R.solve_internal(F)
    assert backward_error(A, X, F) <= TOL
    # one column alone: the same solution to rounding
    x = R.solve_internal(F[:, nrhs // 2])
    assert backward_error(A, x, F[:, nrhs // 2:nrhs // 2 + 1]) <= TOL


# without modes the top levels of this block are not fused; with modes they are
@pytest.mark.parametrize("ngen", [0, 4])
def test_fused_and_unfused_levels(ngen):
    p = parts.hex_block(27, 25, 22, 0.27, 0.25, 0.22, seed=3, n_ext=5)
    print("block 27x25x22, ngen", ngen, flush=True)
    R, A, n1 = solver(p, ngen=ngen)
    for nrhs in (2, 40):
        F = np.random.default_rng(nrhs).normal(0.0, 1.0, (n1, nrhs))
        assert backward_error(A, R.solve_internal(F), F) <= TOL
    # B = -K_ii^-1 K_ib by its definition
    rp, ci, K, _, pe = R.csr()
    full = sp.csr_matrix((K, ci, rp), shape=(len(pe),) * 2)
    eq = np.argsort(pe)
    Kib = full[eq[:n1]][:, eq[n1:]].toarray()
    B = R.B()
    used = np.linalg.norm(Kib, axis=0) > 0  # the rotations of solid external nodes carry no stiffness
    assert backward_error(A, B[:, used], -Kib[:, used]) <= TOL
    assert not np.any(B[:, ~used])
    R.close()


def test_no_boundary_rows_beyond_a_single_front():
    """the smallest tree: one front whose parent is the boundary"""
    p = parts.plate(2, 2, 0.1, 0.1, ext_nodes=[0, 8])
    R, A, n1 = solver(p)
    F = np.random.default_rng(0).normal(0.0, 1.0, (n1, 5))
    assert backward_error(A, R.solve_internal(F), F) <= TOL
    R.close()
