"""Row group of the split-K kernel up to sixteen columns: the smallest whose workgroups have a compute unit each (CPU: the
host-only description of a call)."""
import ctypes

import pytest

from onebitsparsemul_amd import _native


def _rows(token_major, m, n, k, aligned, units):
    plan = (ctypes.c_int * 5)()
    assert _native.lib().onebit_sparse_describe_call(token_major, m, n, k, aligned, units, plan) == 0
    assert plan[0] == 1 and plan[2] == 1  # the split-K kernel, K not split
    return plan[1]


@pytest.mark.parametrize("token_major", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 15, 16])
@pytest.mark.parametrize("units", [32, 256])
def test_rows_at_the_ends_of_each_range(token_major, n, units):
    for rows, last in ((32, 32 * units), (64, 64 * units)):
        assert _rows(token_major, last, n, 2048, 1, units) == rows
        assert _rows(token_major, last + 64, n, 2048, 1, units) == 2 * rows
    assert _rows(token_major, 64, n, 2048, 1, units) == 32
    assert _rows(token_major, 256 * units, n, 2048, 1, units) == 128


@pytest.mark.parametrize("token_major", [0, 1])
@pytest.mark.parametrize("n", [1, 3, 4, 16])
@pytest.mark.parametrize("k", [32, 1024, 1280, 1312])
def test_rows_do_not_depend_on_a_short_k(token_major, n, k):
    for m, rows in ((8192, 32), (8256, 64), (16384, 64), (16448, 128), (20416, 128), (20480, 128)):
        assert _rows(token_major, m, n, k, 1, 256) == rows
