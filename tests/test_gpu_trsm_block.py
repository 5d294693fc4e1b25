"""The 256-row block of the triangular solve at the edges of its fragments and column strips.

Exact cases: integer triangles with powers of two on the diagonal and integer solutions, so that
every intermediate value is an integer or an exact quotient and the solution must come back bit for
bit. Quotients: one-row solves against the IEEE division, ordinary values within one ulp (the
quotient is a once-corrected product with the reciprocal: an error below 1/2 ulp + 2^-50 ulp before
its final rounding), zeros, infinities, NaN and divisors at the ends of the range exactly.
"""
import ctypes as C

import numpy as np
import pytest

import rstsr_amd as rt
from rstsr_amd import abi

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.float64, np.complex64, np.complex128]
ROW, COL, LEFT, RIGHT, UPPER, LOWER, NOTR, NONUNIT, UNIT = 101, 102, 141, 142, 121, 122, 111, 131, 132


@pytest.fixture(scope="module")
def dev():
    return rt.DeviceHIP(0)


def solve(dev, a, b, side, uplo, diag, order=ROW):
    """op: a x = b (left) or x a = b (right); `order` of both buffers."""
    dt = a.dtype
    lay = np.ascontiguousarray if order == ROW else (lambda x: np.ascontiguousarray(x.T))
    ta, tb = rt.asarray(lay(a), device=dev), rt.asarray(lay(b), device=dev)
    one = np.array(1, dtype=dt)
    m, n = b.shape
    abi.check(abi.lib().rstsr_hip_driver_trsm(C.c_void_p(dev._ctx_ptr()), rt._code(dt), 0, order, side, uplo, NOTR, diag,
                                              m, n, one.ctypes.data, ta.as_ptr(), a.shape[0], tb.as_ptr(),
                                              n if order == ROW else m))
    x = tb.to_numpy()
    return x if order == ROW else x.T


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("uplo", [LOWER, UPPER])
def test_exact_solutions(dev, dt, uplo):
    rng = np.random.default_rng(11)
    cx = np.dtype(dt).kind == "c"
    for s, r in [(1, 1), (15, 17), (16, 16), (17, 3), (33, 40), (129, 15), (255, 1), (256, 33), (257, 20), (530, 18)]:
        t = rng.integers(-2, 3, size=(s, s)) + (1j * rng.integers(-2, 3, size=(s, s)) if cx else 0)
        t = np.tril(t, -1) if uplo == LOWER else np.triu(t, 1)
        t = t + np.diag(2.0 ** rng.integers(-2, 3, size=s))
        x = rng.integers(-3, 4, size=(s, r)) + (1j * rng.integers(-3, 4, size=(s, r)) if cx else 0)
        a = t.astype(dt)
        a[(np.triu_indices(s, 1) if uplo == LOWER else np.tril_indices(s, -1))] = np.nan  # not read
        assert np.array_equal(solve(dev, a, (t @ x).astype(dt), LEFT, uplo, NONUNIT), x.astype(dt)), (s, r)
        assert np.array_equal(solve(dev, a, (x.T @ t).astype(dt), RIGHT, uplo, NONUNIT, COL), x.T.astype(dt)), (s, r)
        u = t - np.diag(np.diag(t)) + np.eye(s)
        np.fill_diagonal(a, np.nan)
        assert np.array_equal(solve(dev, a, (u @ x).astype(dt), LEFT, uplo, UNIT), x.astype(dt)), (s, r)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_quotients(dev, dt):
    rng = np.random.default_rng(12)
    fi = np.finfo(dt)
    for d in [3.0, -7.5, 1e-3, fi.max, -fi.tiny, fi.smallest_subnormal, 1.0 / 3.0, np.inf, np.nan, 0.0]:
        b = rng.normal(size=4096) * np.exp2(rng.integers(fi.minexp // 2, fi.maxexp // 2, size=4096))
        b[:8] = [0.0, -0.0, np.inf, -np.inf, np.nan, fi.max, fi.tiny, -fi.tiny]
        b = b.astype(dt)
        with np.errstate(all="ignore"):
            want = b / dt(d)
        got = solve(dev, np.full((1, 1), d, dtype=dt), b[None, :], LEFT, LOWER, NONUNIT)[0]
        plain = np.isfinite(want) & (np.abs(want) >= fi.tiny)
        assert np.array_equal(np.isnan(got), np.isnan(want)), d
        assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)]), d
        assert np.array_equal(got[want == 0], want[want == 0]), d
        assert np.all(np.abs(got[plain] - want[plain]) <= np.spacing(np.abs(want[plain]))), d
        small = np.isfinite(want) & (np.abs(want) < fi.tiny)
        assert np.all(np.abs(got[small] - want[small]) <= fi.smallest_subnormal), d
