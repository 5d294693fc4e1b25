"""Short products with few rows or columns (a thread per output) at the lines of that rule, exact as in
test_gpu_gemm_tile."""
import numpy as np
import pytest

import rstsr_amd as rt
from test_gpu_gemm_tile import DTYPES, embed, ints, product

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return rt.DeviceHIP(0)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("forms", ["c c", "c f", "f c", "f f", "step flip", "flip step"])
def test_exact_products(dev, dt, forms):
    fa, fb = forms.split()
    rng = np.random.default_rng(17)
    for m, n, k in [(2, 2, 1), (16, 17, 16), (16, 33, 17), (17, 40, 16), (500, 3, 5), (5, 700, 2), (256, 259, 9), (257, 300, 16)]:
        a, b = ints(rng, (m, k), dt), ints(rng, (k, n), dt)
        got = (embed(dev, a, fa) % embed(dev, b, fb)).to_numpy()
        assert np.array_equal(got, product(a, b).astype(dt)), (m, n, k)


@pytest.mark.parametrize("dt", DTYPES)
def test_exact_batches(dev, dt):
    """More batches than a grid axis holds, and a broadcast operand."""
    rng = np.random.default_rng(18)
    a, b = ints(rng, (70000, 3, 2), dt), ints(rng, (70000, 2, 4), dt)
    ta, tb = rt.asarray(a, device=dev), rt.asarray(b, device=dev)
    assert np.array_equal((ta % tb).to_numpy(), a @ b)
    assert np.array_equal((ta % tb[0]).to_numpy(), a @ b[0])


@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
def test_complex_symmetric_products_stay_symmetric(dev, dt):
    rng = np.random.default_rng(19)
    x = (rng.normal(size=(9, 12)) + 1j * rng.normal(size=(9, 12))).astype(dt)
    t = rt.asarray(x, device=dev)
    got = (t.transpose() % t).to_numpy()
    assert np.array_equal(got, got.T)


def test_exact_many_small_grouped(dev):
    """More problems than 16 per CU, nearly empty in 128 x 128 tiles: the tuner's tile shape."""
    rng = np.random.default_rng(20)
    probs, want, n0 = [], [], 0
    out = rt.zeros((4300 * 70 * 70,), device=dev)
    for _ in range(4300):
        m, n, k = (int(v) for v in rng.integers(1, 71, size=3))
        a, b = ints(rng, (m, k), np.float64), ints(rng, (k, n), np.float64)
        c = out._view(([m, n], [n, 1], n0))
        probs.append((rt.asarray(a, device=dev), rt.asarray(b, device=dev), c))
        want.append(a @ b)
        n0 += m * n
    rt.gemm_grouped(probs)
    assert np.array_equal(out.to_numpy()[:n0], np.concatenate([w.ravel() for w in want]))
