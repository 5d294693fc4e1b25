"""The complex split GEMM in one run against its three real split products one by one.

The parts are split with the same exponents and the residue products are exact, so C equals
(T1 - T2, (T3 - T1) - T2) of the real products bit for bit, whatever the operands' layouts.
"""
import numpy as np
import pytest

import rstsr_amd as rt

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return rt.DeviceHIP(0)


def wide(rng, shape):
    return rng.normal(size=shape) * np.exp2(rng.integers(-12, 13, size=shape))


def on(dev, x, form):
    """Device tensor with x's values: rows ("c"), columns ("f") or columns of a wider buffer ("s")."""
    if form == "c":
        return rt.asarray(np.ascontiguousarray(x), device=dev)
    if form == "f":
        return rt.asarray(np.ascontiguousarray(x.T), device=dev).transpose()
    buf = np.full((x.shape[0] + 1, 2 * x.shape[1] + 3), 7e77, dtype=x.dtype)
    buf[1:, 1:1 + 2 * x.shape[1]:2] = x
    return rt.asarray(buf, device=dev)[1:, 1:1 + 2 * x.shape[1]:2]


def three(dev, a, b, mode, fa="c", fb="c"):
    p = [rt.matmul(on(dev, np.ascontiguousarray(x), fa), on(dev, np.ascontiguousarray(y), fb), mode=mode).to_numpy()
         for x, y in ((a.real, b.real), (a.imag, b.imag), (a.real + a.imag, b.real + b.imag))]
    with np.errstate(invalid="ignore"):
        return p[0] - p[1], (p[2] - p[0]) - p[1]


@pytest.mark.parametrize("fa,fb", [("c", "c"), ("f", "c"), ("c", "f"), ("f", "f"), ("s", "s")])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (5, 3, 17), (64, 129, 64), (129, 130, 1025), (257, 255, 2049),
                                   (300, 259, 700), (33, 70, 4100), (20, 31, 8200)])
def test_same_bits_as_real_products(dev, m, n, k, fa, fb):
    rng = np.random.default_rng(m + n + k)
    a = wide(rng, (m, k)) + 1j * wide(rng, (m, k))
    b = wide(rng, (k, n)) + 1j * wide(rng, (k, n))
    got = rt.matmul(on(dev, a, fa), on(dev, b, fb), mode="ozaki").to_numpy()
    # the real products' operands keep the layout, which decides the order of the norms' sums
    ra, rb = ("c" if fa == "s" else fa), ("c" if fb == "s" else fb)
    re, im = three(dev, a, b, "ozaki", ra, rb)
    if "s" in (fa, fb):  # other sum orders of the norms: a scale may differ by one binade
        s = np.abs(a).sum(1, keepdims=True) * np.abs(b).max() + 1e-300
        assert np.all(np.abs(got.real - re) <= 1e-14 * s) and np.all(np.abs(got.imag - im) <= 1e-14 * s)
    else:
        assert np.array_equal(got.real, re) and np.array_equal(got.imag, im)


def test_nonfinite(dev):
    """Infinities and NaN appear where the three plain products put them."""
    rng = np.random.default_rng(3)
    for part in (1.0, 1j):
        for bad in (np.inf, np.nan):
            a = rng.normal(size=(40, 70)) + 1j * rng.normal(size=(40, 70))
            b = rng.normal(size=(70, 90)) + 1j * rng.normal(size=(70, 90))
            if part == 1.0:
                a.real[3, 4] = bad
            else:
                b.imag[5, 6] = bad
            got = rt.matmul(rt.asarray(a, device=dev), rt.asarray(b, device=dev), mode="ozaki").to_numpy()
            re, im = three(dev, a, b, "plain")
            for x, y in ((got.real, re), (got.imag, im)):
                assert np.array_equal(np.isnan(x), np.isnan(y)) and np.array_equal(np.isinf(x), np.isinf(y))
                fin = np.isfinite(y)
                assert np.max(np.abs(x[fin] - y[fin])) <= 1e-12


def test_captured(dev):
    """One captured call, launched again on other values."""
    rng = np.random.default_rng(4)
    a = rng.normal(size=(130, 200)) + 1j * rng.normal(size=(130, 200))
    b = rng.normal(size=(200, 140)) + 1j * rng.normal(size=(200, 140))
    ta, tb = rt.asarray(a, device=dev), rt.asarray(b, device=dev)
    rt.matmul(ta, tb, mode="ozaki")  # the workspace grows outside the capture
    with rt.capture(dev) as g:
        out = rt.matmul(ta, tb, mode="ozaki")
    for scale in (1.0, -2.0, 0.5):
        ta.assign(rt.asarray(a * scale, device=dev))
        g.launch()
        want = rt.matmul(rt.asarray(a * scale, device=dev), tb, mode="ozaki").to_numpy()
        assert np.array_equal(out.to_numpy(), want), scale


def test_products_one_by_one_where_memory_is_short():
    """4096^3: the three products at once need 2.1 GB of workspace, one by one 1.65 GB. With 1.8 GB left
    besides the output the call still runs, with the same bits."""
    import ctypes as C

    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()

    def left():
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    n = 4096
    rng = np.random.default_rng(5)
    a = np.resize(rng.normal(size=4099) + 1j * rng.normal(size=4099), (n, n))
    one, two = rt.DeviceHIP(0), rt.DeviceHIP(0)
    t1 = rt.asarray(a, device=one)
    want = rt.matmul(t1, t1, mode="ozaki").to_numpy()
    t2 = rt.asarray(a, device=two)
    one.synchronize()
    out = 16 * n * n
    rt.empty_cache(one)
    hogs = []
    try:
        for _ in range(4):  # the free memory reported lags behind what is freed
            spare = left() - out - (1800 << 20)
            if spare < 32 << 20:
                break
            hogs.append(C.c_void_p())
            assert hip.hipMalloc(C.byref(hogs[-1]), C.c_size_t(spare)) == 0
        assert 1700 << 20 < left() - out < 1900 << 20
        got = rt.matmul(t2, t2, mode="ozaki")
    finally:
        for h in hogs:
            assert hip.hipFree(h) == 0
    assert np.array_equal(got.to_numpy(), want)
