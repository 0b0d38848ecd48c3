"""Modes and reduced matrices over the block widths, boundary sizes and mode
counts where the tall-skinny products change their form (16-column tiles,
one or several row chunks, 16 or 32 rows a wave, one-wave Cholesky factor)."""
import numpy as np
import pytest
import scipy.linalg as sla
import scipy.sparse as sp

from fedempy_amd import gpu, parts

pytestmark = pytest.mark.gpu


def reduced(part, ngen, **opts):
    """eigenvalues, reduced mass matrix and T^T M T of the returned basis T"""
    R = gpu.GpuReducer()
    for k, v in opts.items():
        R.set_option(k, v)
    R.set_part(part)
    z = R.analyze(ngen=ngen)
    R.reduce()
    rp, ci, K, M, pe = R.csr()
    K, M = (sp.csr_matrix((v, ci, rp), shape=(z["neq"],) * 2) for v in (K, M))
    n1 = z["ndof1"]
    eq = np.argsort(pe)  # permuted row of every equation: internal ones first
    K, M = K[eq][:, eq], M[eq][:, eq]
    T = np.zeros((z["neq"], z["ndim"]))
    T[:n1, :z["ndof2"]] = R.B()
    T[n1:, :z["ndof2"]] = np.eye(z["ndof2"])
    if ngen:
        T[:n1, z["ndof2"]:] = R.phi()
    SM, lam = R.reduced()[1], R.eigen()[0]
    R.close()
    return lam, SM, T.T @ (M @ T), K[:n1, :n1], M[:n1, :n1], T[:n1, z["ndof2"]:]


# a sum of n products in any order: n eps of the largest entry
def check_mass(SM, ref):
    assert np.max(np.abs(SM - ref)) <= 1e-11 * np.max(np.abs(ref))


@pytest.mark.parametrize("bs", [1, 3, 15, 16, 17, 32, 33, 48, 64])
def test_block_widths(bs):
    print("block", bs, flush=True)
    p = parts.hex_block(6, 5, 4, 0.06, 0.05, 0.04, seed=3, n_ext=4)
    lam, SM, ref, K, M, phi = reduced(p, 5, lanczosBlock=bs)
    check_mass(SM, ref)
    exact = sla.eigh(K.toarray(), M.toarray(), eigvals_only=True, subset_by_index=[0, 4])
    assert np.max(np.abs(lam - exact) / exact) <= 1e-9


# (fewer than three fixed nodes leave a mechanism, whose mode has no accurate value)
@pytest.mark.parametrize("n_ext,ngen", [(1, 0), (3, 1), (5, 1), (5, 2), (6, 0), (11, 15), (16, 16), (21, 17), (22, 33)])
def test_boundary_and_mode_counts(n_ext, ngen):
    print("external nodes", n_ext, "modes", ngen, flush=True)
    p = parts.hex_block(7, 4, 4, 0.07, 0.04, 0.04, seed=n_ext, n_ext=n_ext)
    lam, SM, ref, K, M, phi = reduced(p, ngen)
    check_mass(SM, ref)
    if ngen:
        exact = sla.eigh(K.toarray(), M.toarray(), eigvals_only=True, subset_by_index=[0, ngen - 1])
        assert np.max(np.abs(lam - exact) / exact) <= 1e-9


# below and above 32,768 rows, with a remainder of the 64- and 128-row tiles
@pytest.mark.parametrize("dims", [(21, 22, 20), (23, 22, 20)])
def test_row_counts(dims):
    print("block of", dims, flush=True)
    p = parts.hex_block(*dims, *(0.01 * d for d in dims), seed=1, n_ext=7)
    lam, SM, ref, K, M, phi = reduced(p, 6)
    check_mass(SM, ref)
    # the Rayleigh quotients of the returned vectors, whose error is the
    # square of the vectors'
    q = np.sum(phi * (K @ phi), axis=0) / np.sum(phi * (M @ phi), axis=0)
    assert np.max(np.abs(lam - q) / q) <= 1e-9


# six equations a node: the consistent mass of beams (sparse product) and the
# lumped one of shells (its diagonal)
@pytest.mark.parametrize("kind", ["beams", "shells"])
@pytest.mark.parametrize("bs", [2, 5, 24, 33, 40, 64])
def test_six_equation_nodes(kind, bs):
    print(kind, "block", bs, flush=True)
    if kind == "beams":
        p = parts.beam_frame(n_el=90, seed=1, n_ext=4)
    else:
        p = parts.plate(9, 7, 0.18, 0.14, ext_nodes=[0, 9, 79])
    lam, SM, ref, K, M, phi = reduced(p, 4, lanczosBlock=bs)
    check_mass(SM, ref)
    q = np.sum(phi * (K @ phi), axis=0) / np.sum(phi * (M @ phi), axis=0)
    assert np.max(np.abs(lam - q) / q) <= 1e-7  # K phi cancels: eps |K| / lambda of a thin part
