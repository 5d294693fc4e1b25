"""Matrix-vector products at the edges of their row groups, vector loads and K splits.

Small integers, so every sum is exact in any order: results equal the integer product bit for bit.
Matrices and vectors are views into NaN-filled buffers (integers: a large filler), so that a
position read past either shows.
"""
import numpy as np
import pytest

import rstsr_amd as rt

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.float64, np.complex64, np.complex128, np.int32, np.int64]
# m, k: single elements, odd tails, one and four waves per row group, splits of k, dot products
SIZES = [(1, 1), (3, 5), (4, 64), (65, 129), (130, 4097), (5000, 33), (16400, 40), (7, 20001), (1, 300001)]


@pytest.fixture(scope="module")
def dev():
    return rt.DeviceHIP(0)


def ints(rng, shape, dt):
    x = rng.integers(-3, 4, size=shape)
    if np.dtype(dt).kind == "c":
        x = x + 1j * rng.integers(-3, 4, size=shape)
    return x.astype(dt)


def filled(shape, dt):
    return np.full(shape, np.nan if np.dtype(dt).kind in "fc" else 1 << 30, dtype=dt)


def matrix(dev, x, form):
    m, n = x.shape
    if form == "c":
        buf = filled((m, n + 3), x.dtype)
        buf[:, 1:1 + n] = x
        return rt.asarray(buf, device=dev)[:, 1:1 + n]
    if form == "f":
        buf = filled((n, m + 3), x.dtype)
        buf[:, 1:1 + m] = x.T
        return rt.asarray(buf, device=dev)[:, 1:1 + m].transpose()
    buf = filled((m, 2 * n + 1), x.dtype)
    buf[:, 1::2] = x[:, ::-1]
    return rt.asarray(buf, device=dev)[:, 1::2].flip(1)


def vector(dev, v, step):
    buf = filled((step * len(v) + 1,), v.dtype)
    buf[1::step][:len(v)] = v
    return rt.asarray(buf, device=dev)[1::step][:len(v)]


def product(a, v):
    if a.dtype.kind == "c":
        ar, ai, br, bi = (p.astype(np.int64) for p in (a.real, a.imag, v.real, v.imag))
        return (ar @ br - ai @ bi) + 1j * (ar @ bi + ai @ br)
    return a.astype(np.int64) @ v.astype(np.int64)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("form", ["c", "f", "step"])
def test_exact(dev, dt, form):
    rng = np.random.default_rng(3)
    for m, k in SIZES:
        a, v = ints(rng, (m, k), dt), ints(rng, (k,), dt)
        want = product(a, v).astype(dt)
        ta = matrix(dev, a, form)
        for step in (1, 2):
            tv = vector(dev, v, step)
            assert np.array_equal((ta % tv).to_numpy(), want), (m, k, step)            # rule 4
            assert np.array_equal((tv % ta.transpose()).to_numpy(), want), (m, k, step)  # rule 3
        if m == 1:
            assert (ta[0] % vector(dev, v, 1)).to_scalar() == want[0]                    # rule 1


@pytest.mark.parametrize("dt", [np.float64, np.complex64])
def test_exact_batches(dev, dt):
    """Batched matrices with one shared vector, and one row per batch (neither folds into one product)."""
    rng = np.random.default_rng(4)
    for b, m, k in [(3, 17, 33), (5, 4, 2050), (70, 2, 9)]:
        a, v = ints(rng, (b, m, k), dt), ints(rng, (k,), dt)
        buf = filled((b, m, k + 1), dt)
        buf[:, :, :k] = a
        got = (rt.asarray(buf, device=dev)[:, :, :k] % rt.asarray(v, device=dev)).to_numpy()
        assert np.array_equal(got, np.stack([product(x, v) for x in a]).astype(dt)), (b, m, k)
        w = ints(rng, (b, k, m), dt)
        x = ints(rng, (b, 1, k), dt)
        got = (rt.asarray(x, device=dev) % rt.asarray(w, device=dev)).to_numpy()
        want = np.stack([product(w[i].T, x[i, 0]) for i in range(b)])[:, None, :].astype(dt)
        assert np.array_equal(got, want), (b, m, k)


@pytest.mark.parametrize("dt", [np.float64, np.float32, np.complex128])
def test_alpha_beta(dev, dt):
    """y = alpha A x + beta y through the strided GEMM entry, without and with a split of k."""
    import ctypes as C

    from rstsr_amd import abi

    rng = np.random.default_rng(5)
    for m, k in [(9, 31), (2, 9000)]:
        a, x, y = ints(rng, (m, k), dt), ints(rng, (k, 1), dt), ints(rng, (m, 1), dt)
        ta, tx, ty = (rt.asarray(z, device=dev) for z in (a, x, y))
        al, be = np.array(2, dtype=dt), np.array(-3, dtype=dt)
        abi.check(abi.lib().rstsr_hip_gemm(C.c_void_p(dev._ctx_ptr()), rt._code(dt), 0, m, 1, k, al.ctypes.data,
                                           ta.as_ptr(), k, 1, tx.as_ptr(), 1, 1, be.ctypes.data, ty.as_ptr(), 1, 1))
        assert np.array_equal(ty.to_numpy()[:, 0], (2 * product(a, x[:, 0]) - 3 * y[:, 0]).astype(dt)), (m, k)


@pytest.mark.parametrize("dt", DTYPES)
def test_hints_by_size_and_sharing(dev, dt):
    """Matrices either side of 40 MB, and one matrix shared by all batches: the same exact results."""
    rng = np.random.default_rng(23)
    es = np.dtype(dt).itemsize
    for m in (1 + (30 << 20) // (1000 * es), 1 + (44 << 20) // (1000 * es)):
        a, x = ints(rng, (m, 1000), dt), ints(rng, 1000, dt)
        want = (a.real.astype(np.int64) @ x.real.astype(np.int64) if np.dtype(dt).kind != "c" else a @ x).astype(dt)
        for form in "cf":
            assert np.array_equal((matrix(dev, a, form) % rt.asarray(x, device=dev)).to_numpy(), want), (m, form)
    a, x = ints(rng, (300, 77), dt), ints(rng, (5, 77, 1), dt)
    got = (rt.asarray(a, device=dev).broadcast_to([5, 300, 77]) % rt.asarray(x, device=dev)).to_numpy()
    assert np.array_equal(got, (a.astype(np.complex128) @ x.astype(np.complex128)).astype(dt) if np.dtype(dt).kind == "c"
                          else (a.astype(np.int64) @ x.astype(np.int64)).astype(dt))
