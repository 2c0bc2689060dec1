"""Saved rows of a batch as the solutions' own arrays: values, and memory in
proportion to what was saved when one trajectory saves far more than the others."""
import tracemalloc

import numpy as np
import pytest

from odemi.api import _trajectory_rows


@pytest.mark.parametrize("n", [0, 1, 3])
@pytest.mark.parametrize("nsaved", [[], [0, 0], [5], [4, 4, 4], [0, 9, 1, 0], [9, 1, 1, 1], [2, 9, 9]])
def test_values(n, nsaved):
    rng = np.random.default_rng(0)
    t, u = rng.random((9, len(nsaved))), rng.random((9, n, len(nsaved)))
    out = _trajectory_rows(t, u, nsaved)
    assert len(out) == len(nsaved)
    for j, (k, (tj, uj)) in enumerate(zip(nsaved, out)):
        assert tj.shape == (k,) and uj.shape == (k, n)
        assert np.array_equal(tj, t[:k, j]) and np.array_equal(uj, u[:k, :, j])
        assert tj.flags.owndata and uj.flags.c_contiguous and not np.shares_memory(uj, u)


def test_one_long_trajectory():
    N, n, rows = 500, 3, 4000
    t, u = np.zeros((rows, N)), np.zeros((rows, n, N))
    nsaved = [20] * N
    nsaved[7] = rows
    tracemalloc.start()
    out = _trajectory_rows(t, u, nsaved)
    peak = tracemalloc.get_traced_memory()[1]
    tracemalloc.stop()
    used = sum(nsaved) * (n + 1) * 8
    # the rows in use, and for each of the arrays its object (well below 1 KB)
    assert peak < used + 2 * N * 1024, (peak, used)
    assert len(out) == N
