"""Values the triangular solve must return exactly: quotients, unit diagonals, sums of many terms."""
import numpy as np
import pytest

import rstsr_amd as rt
from test_gpu_trsm_block import LEFT, LOWER, NONUNIT, UNIT, UPPER, solve

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return rt.DeviceHIP(0)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_quotients_round_as_divisions(dev, dt):
    """A diagonal matrix of 40 divisors: every element is one quotient (b - 0 is b), equal to the IEEE
    division's, subnormal results among them. 40 rows: the block kernel."""
    rng = np.random.default_rng(21)
    fi = np.finfo(dt)
    s, r = 40, 3000
    d = (rng.uniform(1, 2, size=s) * np.exp2(rng.integers(-20, 21, size=s))).astype(dt)
    d[::7] = -d[::7]
    lo = np.exp2(rng.integers(fi.minexp - fi.nmant, fi.minexp + 25, size=(s, r)).astype(np.float64))
    b = rng.uniform(-2, 2, size=(s, r)) * np.where(rng.random((s, r)) < 0.5, 1.0, lo)
    b = b.astype(dt)
    want = b / d[:, None]
    assert np.any((want != 0) & (np.abs(want) < fi.tiny)) and np.all(np.isfinite(want))
    assert np.array_equal(solve(dev, np.diag(d), b, LEFT, LOWER, NONUNIT), want)


@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
@pytest.mark.parametrize("uplo", [LOWER, UPPER])
def test_unit_diagonal_keeps_non_finite_parts(dev, dt, uplo):
    """A unit diagonal divides nothing: rows that nothing is subtracted from come back as they are,
    each part's infinities and NaN to itself."""
    parts = [3.0, -0.5, np.inf, -np.inf, np.nan]
    b0 = np.array([complex(re, im) for re in parts for im in parts], dtype=dt)
    for s in (1, 20, 40):
        b = np.ones((s, b0.size), dtype=dt)
        first = 0 if uplo == LOWER else s - 1
        b[first] = b0
        a = np.zeros((s, s), dtype=dt)
        np.fill_diagonal(a, np.nan)  # not read
        got = solve(dev, a, b, LEFT, uplo, UNIT)[first]
        for g, w in ((got.real, b0.real), (got.imag, b0.imag)):
            assert np.array_equal(g, w, equal_nan=True), s


@pytest.mark.parametrize("dt", [np.float32, np.float64, np.complex64, np.complex128])
@pytest.mark.parametrize("uplo", [LOWER, UPPER])
def test_small_updates_add_up_before_they_are_subtracted(dev, dt, uplo):
    """240 updates of u / 2 each (u: the unit roundoff) of one row: 1 - u / 2 rounds to 1, their sum
    120 u is exact, and so is 1 - 120 u."""
    s, m = 256, 240
    u = np.finfo(dt).epsneg
    a = np.eye(s, dtype=dt)
    b = np.ones((s, 20), dtype=dt)
    want = b.copy()
    if uplo == LOWER:
        a[-1, :m] = u / 2
        want[-1] = 1 - 120 * u
    else:
        a[0, -m:] = u / 2
        want[0] = 1 - 120 * u
    assert np.array_equal(solve(dev, a, b, LEFT, uplo, NONUNIT), want)


@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
@pytest.mark.parametrize("s", [5, 40])
def test_complex_quotients(dev, dt, s):
    """Diagonal solves on both kernels against extended precision, divisors of every magnitude. The parts
    of a conj(b) are off by 2 u |a||b|, |b|^2 and the quotient by 2 u and u: 2 sqrt(2) u + 3 u < 6 u of |a / b|."""
    rng = np.random.default_rng(25)
    u = np.finfo(dt).eps / 2
    e = 40 if dt == np.complex64 else 300
    d = (rng.normal(size=s) + 1j * rng.normal(size=s)) * np.exp2(rng.integers(-e, e + 1, size=s))
    d[::3] = d[::3].real  # one part zero
    d, b = d.astype(dt), (rng.normal(size=(s, 700)) + 1j * rng.normal(size=(s, 700))).astype(dt)
    want = b.astype(np.clongdouble) / d.astype(np.clongdouble)[:, None]
    got = solve(dev, np.diag(d), b, LEFT, LOWER, NONUNIT)
    assert np.all(np.abs(got - want) <= 6 * u * np.abs(want))
