"""B, modes, solutions, recovered displacements, load vectors and gravity
forces on their way between the caller and the device, which goes by pieces of
65,536 values: whole columns, several or one, with a remainder, and rows of 16
columns where a column is longer than a sixteenth of a piece, or than a piece."""
import numpy as np
import pytest
import scipy.sparse as sp

from fedempy_amd import gpu, parts
from test_solve_rhs_gpu import TOL, backward_error

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["1479 rows", "5544 rows", "71844 rows"])
def part(request):
    p = {"1479 rows": lambda: parts.hex_block(16, 5, 4, 0.16, 0.05, 0.04, seed=6, n_ext=17),
         "5544 rows": lambda: parts.plate(30, 29, 0.3, 0.29, ext_nodes=[0, 29, 870, 899, 450, 455]),
         "71844 rows": lambda: parts.plate(112, 105, 1.12, 1.05, ext_nodes=[0, 105, 11000, 11977])}[request.param]()
    R = gpu.GpuReducer()
    R.set_part(p)
    z = R.analyze(ngen=3)
    R.reduce()
    assert z["ndof1"] == int(request.param.split()[0])
    rp, ci, K, M, pe = R.csr()
    eq = np.argsort(pe)
    K, M = (sp.csr_matrix((v, ci, rp), shape=(z["neq"],) * 2)[eq][:, eq] for v in (K, M))
    yield R, z, K, M, R.B()
    R.close()


def test_recovery_matrix_and_gravity(part):
    R, z, K, M, B = part
    n1 = z["ndof1"]
    Kib = K[:n1][:, n1:].toarray()
    on = np.any(Kib, axis=0)  # (the rotations of a solid's external node couple to nothing)
    assert backward_error(K[:n1][:, :n1], B[:, on], -Kib[:, on]) <= TOL and not B[:, ~on].any()
    phi, lam = R.phi(), R.eigen()[0]
    P = phi[:, :3]
    assert np.max(np.abs(P.T @ (M[:n1][:, :n1] @ P) - np.eye(3))) <= 1e-9
    # in the norm and within a hundred times the limit of the iteration's own test
    E = R.solve_internal(np.asfortranarray(M[:n1][:, :n1] @ P)) * lam[:3] - P
    assert np.max(np.einsum("ij,ij->j", E, M[:n1][:, :n1] @ E)) <= 1e-18
    sam = R.sam()
    a = np.zeros((z["neq"], 3))
    for n in range(z["nnod"]):
        for c in range(3):
            e = sam["meqn"][sam["madof"][n] - 1 + c]
            if e > 0:
                a[e - 1, c] = 1.0
    g = np.full((n1, 3), np.nan, order="F")
    R._check(R.lib.fgpu_get_gravity_internal(R.h, gpu._ptr(g)), "fgpu_get_gravity_internal")
    ref = (M @ a)[:n1]
    assert np.max(np.abs(g - ref)) <= 1e-13 * np.abs(ref).max()


@pytest.mark.parametrize("nrhs", [1, 11, 12, 16, 17, 44, 45, 64, 90])
def test_solutions_recovery_and_loads(part, nrhs):
    R, z, K, _, B = part
    n1, n2, neq, nd = z["ndof1"], z["ndof2"], z["neq"], z["ndim"]
    rng = np.random.default_rng(nrhs)
    F = np.asfortranarray(rng.normal(size=(neq, nrhs)))
    Fi, Ub = np.asfortranarray(F[:n1]), np.asfortranarray(rng.normal(size=(n2, nrhs)))
    X = R.solve_internal(Fi)
    assert backward_error(K[:n1][:, :n1], X, Fi) <= TOL

    def recover(ub, fi):
        u = np.full((n1, nrhs), np.nan, order="F")
        R._check(R.lib.fgpu_recover(R.h, nrhs, None if ub is None else gpu._ptr(ub), None if fi is None else gpu._ptr(fi),
                                    gpu._ptr(u)), "fgpu_recover")
        return u

    assert np.array_equal(recover(None, Fi), X)
    U = recover(Ub, None)
    # sums of n2 products
    assert np.max(np.abs(U - B @ Ub)) <= 1e-12 * np.abs(B).max() * np.abs(Ub).sum(0).max()
    assert np.array_equal(recover(Ub, Fi), U + X)
    fred = np.full((nd, nrhs), np.nan, order="F")
    R._check(R.lib.fgpu_reduce_loads(R.h, nrhs, gpu._ptr(F), gpu._ptr(fred)), "fgpu_reduce_loads")
    pos = np.asarray(R.sam()["dofPosIn2"])[:n2] - 1
    ref = np.vstack([(F[n1:] + B.T @ F[:n1])[pos], R.phi()[:, :3].T @ F[:n1]])
    # sums of neq products
    assert np.max(np.abs(fred[:n2 + 3] - ref)) <= 1e-12 * max(1.0, np.abs(B).max()) * np.abs(F).sum(0).max()
    assert not fred[n2 + 3:].any()
