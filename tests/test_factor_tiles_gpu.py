"""Diagonal blocks of the factorisation at the edges of their 16- and
64-column tiles: beam chains of one front (6 pivot columns per internal
node) against the oracle, at the FP64 path's 1e-10."""
import numpy as np
import pytest

from fedempy_amd import gpu, parts
from oracle import reducer as orc

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def chain(k, straight=False):
    """k internal nodes between two external ones; zig-zag unless straight."""
    n = np.arange(k + 2)
    y = np.zeros(k + 2) if straight else 0.02 * (n % 3)
    p = dict(xyz=np.stack([0.05 * n, y, 0.5 * y], 1), status=np.where((n == 0) | (n == k + 1), 1, 0).astype(np.int32),
             melcon=np.full(k + 1, 11, np.int32), mpmnpc=(1 + 2 * np.arange(k + 2)).astype(np.int32),
             mmnpc=np.stack([n[:-1], n[1:]], 1).ravel().astype(np.int32) + 1,
             eprop=parts._stiff_beam_props(k + 1, v=(0.0, 0.0, 1.0)))
    return p


# pivot columns 6 k: inside one 16-column tile, just past it, at 48 and 60
# (the last tile partly filled), past 64 (two panels), 126 and 144
@pytest.mark.parametrize("k", [1, 2, 3, 5, 8, 10, 11, 16, 21, 24])
@pytest.mark.parametrize("mixed", [False, True])
def test_chain_matches_oracle(k, mixed):
    p = chain(k)
    print("chain", k, "mixed" if mixed else "fp64", flush=True)
    R = gpu.GpuReducer()
    if mixed:
        R.set_option("mixedPrecision", 1)
    R.set_part(p)
    R.analyze(vgi=True)
    R.reduce()
    SK, SM, G = R.reduced()
    o = orc.reduce(p, want_vgi=True)
    tol = 1e-8 if mixed else 1e-10  # the two paths' tolerances against the oracle
    for a, b in ((SK, o["SK"]), (SM, o["SM"]), (G, o["G"]), (R.B(), o["B"]), (R.vgi(), o["vgi"])):
        assert rel(a, b) <= tol


# a node without torsional stiffness: one zero pivot, in another tile each time
@pytest.mark.parametrize("node", [1, 4, 9, 12, 20])
def test_zero_pivot_in_any_tile(node):
    p = chain(22, straight=True)
    p["eprop"][[node - 1, node], 7] = 0.0  # J of the elements on both sides
    print("zero torsion at node", node, flush=True)
    R = gpu.GpuReducer()
    R.set_part(p)
    R.analyze()
    R.reduce()
    (neg, ntrue, nred), sing = R.pivots()
    assert (neg, ntrue, nred) == (0, 1, 0)
    assert [(s[0], s[1], s[3]) for s in sing] == [(node + 1, 4, 1)]
    s = orc.sam_numbering(p)
    K = orc.assemble(p, s)[0].toarray()
    i1, i2 = s["meqn1"] - 1, s["meqn2"] - 1
    S = K[np.ix_(i2, i2)] - K[np.ix_(i2, i1)] @ np.linalg.pinv(K[np.ix_(i1, i1)], rcond=1e-13) @ K[np.ix_(i1, i2)]
    assert rel(R.reduced()[0], S) <= 1e-9  # the hinged blocks' tolerance
