"""Triangular solves of few rows and many columns (a thread per column), at the lines between the two
kernels. Integer triangles with powers of two on the diagonal and integer solutions: every
intermediate value is exact, so the solution must come back bit for bit."""
import numpy as np
import pytest

import rstsr_amd as rt
from test_gpu_trsm_block import COL, DTYPES, LEFT, LOWER, NONUNIT, RIGHT, UNIT, UPPER, solve

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return rt.DeviceHIP(0)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("uplo", [LOWER, UPPER])
def test_exact_solutions(dev, dt, uplo):
    rng = np.random.default_rng(31)
    cx = np.dtype(dt).kind == "c"
    # rows, columns: one, part of a block of columns, either side of 8 and 32 rows, a block of 256
    # rows and 14 more
    for s, r in [(1, 1), (2, 65), (8, 129), (9, 10001), (31, 33001), (32, 33001), (33, 33001), (270, 16001)]:
        t = rng.integers(-2, 3, size=(s, s)) + (1j * rng.integers(-2, 3, size=(s, s)) if cx else 0.0)
        t = np.tril(t, -1) if uplo == LOWER else np.triu(t, 1)
        t = t + np.diag(2.0 ** rng.integers(-2, 3, size=s))
        x = rng.integers(-3, 4, size=(s, r)) + (1j * rng.integers(-3, 4, size=(s, r)) if cx else 0.0)
        a = t.astype(dt)
        a[(np.triu_indices(s, 1) if uplo == LOWER else np.tril_indices(s, -1))] = np.nan  # not read
        assert np.array_equal(solve(dev, a, (t @ x).astype(dt), LEFT, uplo, NONUNIT), x.astype(dt)), (s, r)
        assert np.array_equal(solve(dev, a, (x.T @ t).astype(dt), RIGHT, uplo, NONUNIT, COL), x.T.astype(dt)), (s, r)
        u = t - np.diag(np.diag(t)) + np.eye(s)
        np.fill_diagonal(a, np.nan)
        assert np.array_equal(solve(dev, a, (u @ x).astype(dt), LEFT, uplo, UNIT), x.astype(dt)), (s, r)
