"""Matrix-core tile GEMM at the edges of its tiles, chunks and K slices.

Operands are small integers, so every sum is exact in the element type whatever its order: results
must equal the integer product bit for bit. Operands are views into buffers whose every other
element is NaN, so a position read past a row, a slice or a matrix shows in the result.
"""
import numpy as np
import pytest

import rstsr_amd as rt

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.float64, np.complex64, np.complex128]
# m, n, k: one element, either side of the 16-byte chunks, of the 32 / 64 / 128 tiles and of the
# 128-byte K slices; the last rows are split along K
SIZES = [(1, 1, 1), (3, 2, 5), (31, 33, 7), (32, 64, 32), (63, 65, 33), (64, 64, 64), (65, 127, 31), (129, 130, 66),
         (200, 257, 97), (1, 300, 129), (300, 1, 130), (37, 45, 2049), (64, 128, 4096)]


@pytest.fixture(scope="module")
def dev():
    return rt.DeviceHIP(0)


def ints(rng, shape, dt):
    x = rng.integers(-4, 5, size=shape).astype(np.float64)
    if np.dtype(dt).kind == "c":
        x = x + 1j * rng.integers(-4, 5, size=shape)
    return x.astype(dt)


def embed(dev, x, form):
    """x as a device view inside a NaN buffer: c (rows padded), f (columns padded), step (no unit
    stride), flip (unit stride backwards)."""
    m, n = x.shape
    nan = np.array(np.nan, dtype=x.dtype)
    if form == "c":
        buf = np.full((m + 1, n + 3), nan)
        buf[:m, 1:1 + n] = x
        return rt.asarray(buf, device=dev)[:m, 1:1 + n]
    if form == "f":
        buf = np.full((n + 1, m + 3), nan)
        buf[:n, 2:2 + m] = x.T
        return rt.asarray(buf, device=dev)[:n, 2:2 + m].transpose()
    if form == "step":
        buf = np.full((2 * m, 2 * n + 1), nan)
        buf[::2, 1::2] = x
        return rt.asarray(buf, device=dev)[::2, 1::2]
    buf = np.full((m, n + 2), nan)
    buf[:, 1:1 + n] = x[:, ::-1]
    return rt.asarray(buf, device=dev)[:, 1:1 + n].flip(1)


def product(a, b):
    if a.dtype.kind == "c":
        ar, ai, br, bi = (p.astype(np.int64) for p in (a.real, a.imag, b.real, b.imag))
        return (ar @ br - ai @ bi) + 1j * (ar @ bi + ai @ br)
    return (a.astype(np.int64) @ b.astype(np.int64)).astype(np.float64)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("forms", ["cc", "cf", "fc", "ff", "step c", "c step", "flip f", "f flip"])
def test_exact_products(dev, dt, forms):
    fa, fb = forms.split() if " " in forms else forms
    rng = np.random.default_rng(7)
    for m, n, k in SIZES:
        a, b = ints(rng, (m, k), dt), ints(rng, (k, n), dt)
        got = (embed(dev, a, fa) % embed(dev, b, fb)).to_numpy()
        assert np.array_equal(got, product(a, b).astype(dt)), (m, n, k)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("form", ["c", "f"])
def test_exact_symmetric_products(dev, dt, form):
    """x^T x of one buffer: the lower tiles and their mirror, also with K split."""
    rng = np.random.default_rng(8)
    for k, n in [(5, 3), (33, 66), (100, 129), (2050, 45)]:
        x = ints(rng, (k, n), dt)
        t = embed(dev, x, form)
        got = (t.transpose() % t).to_numpy()
        assert np.array_equal(got, product(x.T, x).astype(dt)), (k, n)


@pytest.mark.parametrize("dt", [np.float64, np.complex128])
def test_exact_grouped(dev, dt):
    """Uneven problems of every operand form in one call; the outputs' padding stays NaN."""
    rng = np.random.default_rng(9)
    probs, refs = [], []
    forms = ["cc", "cf", "fc", "ff", ("step", "c"), ("flip", "f")]
    for i, (m, n, k) in enumerate(SIZES * 2):
        fa, fb = forms[i % len(forms)]
        a, b = ints(rng, (m, k), dt), ints(rng, (k, n), dt)
        out = rt.asarray(np.full((m + 1, n + 1), np.nan, dtype=dt), device=dev)
        probs.append((embed(dev, a, fa), embed(dev, b, fb), out[:m, :n]))
        refs.append((product(a, b).astype(dt), out, m, n))
    rt.gemm_grouped(probs)
    for ref, out, m, n in refs:
        got = out.to_numpy()
        assert np.array_equal(got[:m, :n], ref), (m, n)
        assert np.isnan(got[m:]).all() and np.isnan(got[:, n:]).all()
