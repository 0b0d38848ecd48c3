"""Load vectors, solutions, B and modes between the callers' order and the
device's, over column counts at the edges of the 16-column tiles and of the
64-column chunks of the recovery."""
import numpy as np
import pytest

from fedempy_amd import gpu, parts

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def reduced():
    R = gpu.GpuReducer()
    R.set_part(parts.hex_block(7, 5, 4, 0.07, 0.05, 0.04, seed=6, n_ext=5))
    z = R.analyze(ngen=4)
    R.reduce()
    yield R, z, R.B(), R.phi(), R.sam()
    R.close()


def close(a, b, scale):
    # sums of some hundred products in another order
    return np.max(np.abs(a - b), initial=0.0) <= 1e-12 * scale


@pytest.mark.parametrize("nrhs", [1, 15, 16, 17, 63, 64, 65, 130])
def test_loads_and_recovery(reduced, nrhs):
    R, z, B, phi, sam = reduced
    n1, n2, neq = z["ndof1"], z["ndof2"], z["neq"]
    rng = np.random.default_rng(nrhs)
    F = np.asfortranarray(rng.normal(size=(neq, nrhs)))
    Ub = np.asfortranarray(rng.normal(size=(n2, nrhs)))
    e1, e2 = np.asarray(sam["meqn1"]) - 1, np.asarray(sam["meqn2"]) - 1
    Fi = np.asfortranarray(F[e1])
    X = R.solve_internal(Fi)
    ui = np.zeros((n1, nrhs), order="F")
    for ub, fi, ref in ((Ub, None, B @ Ub), (None, Fi, X), (Ub, Fi, B @ Ub + X), (None, None, 0 * X)):
        ui[:] = np.nan
        R._check(R.lib.fgpu_recover(R.h, nrhs, None if ub is None else gpu._ptr(ub), None if fi is None else gpu._ptr(fi),
                                    gpu._ptr(ui)), "fgpu_recover")
        assert close(ui, ref, np.abs(B).max() * np.abs(Ub).sum(0).max() + np.abs(X).max())
    fred = np.full((z["ndim"], nrhs), np.nan, order="F")
    R._check(R.lib.fgpu_reduce_loads(R.h, nrhs, gpu._ptr(F), gpu._ptr(fred)), "fgpu_reduce_loads")
    r2 = F[e2] + B.T @ F[e1]
    pos = np.asarray(sam["dofPosIn2"])[:n2] - 1
    ref = np.vstack([r2[pos], phi.T @ F[e1]])
    scale = max(np.abs(B).max(), np.abs(phi).max(), 1.0) * np.abs(F).sum(0).max()
    assert close(fred[:n2 + 4], ref, scale) and not fred[n2 + 4:].any()
