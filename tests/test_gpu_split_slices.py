"""The split GEMM's 256 x 256 tile over every short sequence of K slices and over more than one K chunk.

Small integers split without rounding, so the product equals the integer product exactly.
"""
import numpy as np
import pytest

import rstsr_amd as rt

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return rt.DeviceHIP(0)


# one slice, two, three, ... of 128; 65664 and 131200: a second and a third chunk, added to the residues
@pytest.mark.parametrize("k", [1, 127, 128, 129, 256, 257, 384, 385, 640, 65536, 65664, 131200])
@pytest.mark.parametrize("m,n", [(257, 257), (300, 515)])
def test_exact(dev, m, n, k):
    rng = np.random.default_rng(k)
    a = rng.integers(-99, 100, size=(m, k)).astype(np.float64)
    b = rng.integers(-99, 100, size=(k, n)).astype(np.float64)
    got = rt.matmul(rt.asarray(a, device=dev), rt.asarray(b, device=dev), mode="ozaki").to_numpy()
    assert np.array_equal(got, a @ b)  # sums below 2^53: exact in any order


@pytest.mark.parametrize("b,m,n,k", [(1, 2049, 1793, 200), (40, 260, 270, 130)])
def test_moduli_in_sequence(dev, b, m, n, k):
    """Several moduli per block: the slices run on across the residue epilogues."""
    rng = np.random.default_rng(b)
    x = rng.integers(-99, 100, size=(b, m, k)).astype(np.float64)
    y = rng.integers(-99, 100, size=(b, k, n)).astype(np.float64)
    got = rt.matmul(rt.asarray(x, device=dev), rt.asarray(y, device=dev), mode="ozaki").to_numpy()
    assert np.array_equal(got, x @ y)
