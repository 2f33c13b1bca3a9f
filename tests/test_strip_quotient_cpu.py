"""The W application's element -> (row, column) split, as the kernel computes it in 32 bits:
exact for every strip that a plan may hold (fewer than 2^22 columns, elements and two
columns more below 2^31)."""
import numpy as np
import pytest


def _split(e, rows):
    f = np.float32
    j = (e.astype(f) * (f(1) / f(rows))).astype(np.int64)
    j = np.where(j * rows > e, j - 1, np.where((j + 1) * rows <= e, j + 1, j))
    assert (np.abs((j + 1) * rows) < 2**31).all()
    return j


@pytest.mark.parametrize("cols_log2", [1, 11, 16, 20, 22])
def test_quotient_is_exact(cols_log2):
    rng = np.random.default_rng(cols_log2)
    for _ in range(100):
        cols = int(rng.integers(2**(cols_log2 - 1), 2**cols_log2))
        rows = int(rng.integers(1, max(2, (2**31 - 1 - 2048) // (cols + 2))))
        n = rows * cols
        edge = rng.integers(0, cols, 4000) * rows
        e = np.concatenate([rng.integers(0, n, 4000), edge, edge + rows - 1, edge + rows // 2, [0, n - 1]])
        assert np.array_equal(_split(e, rows), e // rows), (rows, cols)
