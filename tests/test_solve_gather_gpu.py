"""Solves over trees whose fronts have more than two children, one or two of
them, beside the right-hand side counts up to which the products gather their
source rows."""
import numpy as np
import pytest

from fedempy_amd import parts
from test_solve_rhs_gpu import TOL, backward_error, solver

pytestmark = pytest.mark.gpu


def star(arms, n):
    """arms of n beam elements from one internal joint, the tips external"""
    xyz, conn, ext = [[0.0, 0.0, 0.0]], [], []
    for a in range(arms):
        d = np.array([np.cos(2 * np.pi * (a + 0.3) / arms), np.sin(2 * np.pi * (a + 0.3) / arms), 0.1 * a])
        for i in range(n):
            conn.append(np.array([0 if i == 0 else len(xyz) - 1, len(xyz)]))
            xyz.append(list(d * (i + 1) / n))
        ext.append(len(xyz) - 1)
    status = np.zeros(len(xyz), np.int32)
    status[ext] = 1
    props = np.tile(parts.beam_frame(60)["eprop"][0], (len(conn), 1))
    props[:, 8:11] = [0.0, 0.0, 1.0]
    return parts._finish(np.array(xyz), status, np.full(len(conn), 11, np.int32), conn, props)


@pytest.mark.parametrize("make", [lambda: star(8, 40), lambda: parts.beam_frame(450, seed=2, n_ext=7),
                                  lambda: parts.plate(33, 29, 0.33, 0.29, ext_nodes=[0, 29, 990, 1019])],
                         ids=["star", "frame", "plate"])
@pytest.mark.parametrize("mixed", [False, True])
def test_gathered_sources(make, mixed):
    print("mixed" if mixed else "fp64", flush=True)
    R, A, n1 = solver(make(), mixed=mixed)
    kids = np.bincount(np.asarray(R.supernodes()["parent"])[:-1])
    print("children per front", np.bincount(kids), flush=True)
    for nrhs in (1, 7, 16, 17, 32, 33, 48):
        F = np.random.default_rng(nrhs).normal(0.0, 1.0, (n1, nrhs))
        assert backward_error(A, R.solve_internal(F), F) <= TOL
    R.close()
