"""Parts of different sizes in turn on one handle, and handles made and closed
in turn: the buffers, plans and pinned memory that one part leaves serve the
next, and the results are those of a handle of its own, bit for bit.  The
parts' arrays lie on both sides of the pieces (512 KB) in which they are
uploaded."""
import threading

import numpy as np
import pytest

from fedempy_amd import gpu, parts

pytestmark = pytest.mark.gpu

PARTS = [
    (lambda: parts.hex_block(9, 8, 7, 0.09, 0.08, 0.07, seed=1, n_ext=5), 4),
    (lambda: parts.plate(75, 71, 0.75, 0.71, ext_nodes=[0, 71]), 0),
    (lambda: parts.beam_frame(60, seed=3, n_ext=4), 3),
    (lambda: parts.hex_block(20, 17, 15, 0.2, 0.17, 0.15, seed=4, n_ext=6), 6),
    (lambda: parts.plate(20, 10, 0.2, 0.1, ext_nodes=[0, 10]), 2),
]


def results(R, make, ngen):
    R.set_part(make())
    z = R.analyze(ngen=ngen)
    R.reduce()
    F = np.random.default_rng(7).normal(size=(z["ndof1"], 5))
    return [*R.reduced(), R.B(), R.solve_internal(F)] + ([R.eigen()[0], R.phi()] if ngen else [])


@pytest.fixture(scope="module")
def alone():
    out = []
    for make, ngen in PARTS:
        R = gpu.GpuReducer()
        out.append(results(R, make, ngen))
        R.close()
    return out


def same(a, b):
    return len(a) == len(b) and all(np.array_equal(x, y) for x, y in zip(a, b))


def test_parts_in_turn_on_one_handle(alone):
    R = gpu.GpuReducer()
    for q in (0, 1, 2, 3, 4, 3, 0, 1, 1):
        print("part", q, flush=True)
        assert same(results(R, *PARTS[q]), alone[q])
    R.close()


def test_handles_in_turn_on_threads(alone):
    bad = []

    def work(first):
        for q in range(first, first + 6):
            R = gpu.GpuReducer()
            if not same(results(R, *PARTS[q % 5]), alone[q % 5]):
                bad.append(q % 5)
            R.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
