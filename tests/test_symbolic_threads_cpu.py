"""Fronts of parts on both sides of the size from which the ordering and the
front lists are made by several threads (4000 nodes)."""
import numpy as np
import pytest

from fedempy_amd import gpu, parts


@pytest.mark.parametrize("make", [
    lambda: parts.plate(62, 62, 0.62, 0.62, ext_nodes=[0, 62]),  # 3969 nodes
    lambda: parts.plate(63, 62, 0.63, 0.62, ext_nodes=[0, 63]),  # 4032 nodes
    lambda: parts.hex_block(21, 17, 14, 0.21, 0.17, 0.14, seed=4, n_ext=9),
])
def test_fronts_are_closed_and_repeatable(make):
    part, out = make(), []
    for _ in range(3):
        R = gpu.GpuReducer()
        R.set_part(part)
        z = R.analyze()
        out.append(R.supernodes())
        R.close()
    s = out[0]
    for o in out[1:]:
        assert all(np.array_equal(np.asarray(o[k]), np.asarray(s[k])) for k in s)
    assert np.array_equal(np.sort(s["perm_to_eq"]), np.arange(z["neq"]))
    ptr = np.concatenate([[0], np.cumsum(s["nrow"])])
    rows = [s["rows"][a:b] for a, b in zip(ptr[:-1], ptr[1:])]
    for q, r in enumerate(rows):
        assert np.all(np.diff(r) > 0)
        assert np.array_equal(r[:s["ncol"][q]], s["col0"][q] + np.arange(s["ncol"][q]))
        if s["parent"][q] >= 0:  # a child's update rows are rows of its parent
            assert np.all(np.isin(r[s["ncol"][q]:], rows[s["parent"][q]]))
