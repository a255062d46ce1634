"""Cells as the model keeps them, where the indices reach far beyond the number
of cells: order, sums of duplicates, and time and memory that follow the cells
(counts per index took seconds and gigabytes at 2^31; a second is 100 times what
60 cells need)."""
import time

import numpy as np
import pytest

from macau_amd import _lib
from macau_amd._lib import check, ptr

TOP = 2147483647


def _test_data(idx, vals, dims):
    L = _lib.lib()
    h = L.macau_make_fixed(len(dims), 4, 1.0)
    assert h, _lib.last_error()
    try:
        ix, v = np.asfortranarray(idx, dtype=np.int32), np.ascontiguousarray(vals, dtype=np.float64)
        d = np.array(dims, dtype=np.int32)
        t0 = time.monotonic()
        check(L.macau_set_relation_data_test(h, ptr(ix), len(dims), ptr(v), len(v), ptr(d)))
        assert time.monotonic() - t0 < 1.0
        n = L.macau_get_test_nonzeros(h)
        out = np.zeros((n, len(dims) + 1), order="F")
        check(L.macau_get_test_data(h, ptr(out)))
        return np.array(out)
    finally:
        L.macau_free(h)


@pytest.mark.parametrize("dims", [(7, 5), (TOP, 5), (7, TOP), (TOP, TOP)])
def test_matrix_test_cells_of_any_size(dims):
    rng = np.random.default_rng(3)
    top = [min(d, 1000) for d in dims]
    idx = np.stack([rng.integers(0, t, 60) for t in top], 1)
    idx[::7] = idx[3]  # duplicates
    idx[5] = [d - 1 for d in dims]
    vals = rng.standard_normal(60)
    got = _test_data(idx, vals, dims)
    order = sorted(range(60), key=lambda e: (idx[e, 1], idx[e, 0]))
    want = {}
    for e in order:
        k = (int(idx[e, 0]), int(idx[e, 1]))
        want[k] = want.get(k, 0.0) + vals[e]
    np.testing.assert_array_equal(got[:, :2], np.array(list(want), dtype=np.float64))
    np.testing.assert_array_equal(got[:, 2], np.array(list(want.values())))


@pytest.mark.parametrize("first", [9, TOP])
def test_tensor_test_cells_of_any_size(first):
    rng = np.random.default_rng(4)
    idx = np.stack([rng.integers(0, min(first, 900), 50), rng.integers(0, 4, 50), rng.integers(0, 6, 50)], 1)
    idx[8, 0] = first - 1
    vals = rng.standard_normal(50)
    got = _test_data(idx, vals, (first, 4, 6))
    order = np.argsort(idx[:, 0], kind="stable")
    np.testing.assert_array_equal(got[:, :3], idx[order])
    np.testing.assert_array_equal(got[:, 3], vals[order])
