"""Reductions at the edges of their lane groups, packs and parts of the reduced range.

Integer-valued operands, so that every result is exact in any order and equals numpy's bit for bit.
Inputs are views into larger buffers of another value: a position read past a view shows.
"""
import numpy as np
import pytest

import rstsr_amd as rt

pytestmark = pytest.mark.gpu

DTYPES = [np.int32, np.float32, np.float64, np.complex64, np.complex128, np.int64]
FILL = 777777


@pytest.fixture(scope="module")
def dev():
    return rt.DeviceHIP(0)


def ints(rng, shape, dt):
    x = rng.integers(-9, 10, size=shape)
    if np.dtype(dt).kind == "c":
        x = x + 1j * rng.integers(-9, 10, size=shape)
    return x.astype(dt)


def inside(dev, x, lead):
    """x as a contiguous view `lead` elements into a filled device buffer."""
    buf = np.full(x.size + lead + 5, FILL, dtype=x.dtype)
    buf[lead:lead + x.size] = x.reshape(-1)
    stride = [int(np.prod(x.shape[i + 1:])) for i in range(x.ndim)]
    return rt.asarray(buf, device=dev)._view((list(x.shape), stride, lead))


def mid(dev, x):
    """x as a strided view inside a filled device buffer, one position off every edge."""
    buf = np.full([n + 2 for n in x.shape], FILL, dtype=x.dtype)
    sl = tuple(slice(1, n + 1) for n in x.shape)
    buf[sl] = x
    return rt.asarray(buf, device=dev)[sl]


@pytest.mark.parametrize("dt", DTYPES[:3] + DTYPES[5:])
@pytest.mark.parametrize("rows,cols", [(40000, 1), (40000, 3), (40000, 17), (33001, 63), (33001, 257), (33001, 511),
                                       (9001, 513), (257, 1025), (1, 70001)])
def test_row_groups(dev, dt, rows, cols):
    rng = np.random.default_rng(cols)
    x = ints(rng, (rows, cols), dt)
    for t in (inside(dev, x, 0), inside(dev, x, 1), mid(dev, x)):
        assert np.array_equal(t.sum_axes([1]).to_numpy(), x.sum(axis=1, dtype=x.dtype))
        assert np.array_equal(t.max_axes([1]).to_numpy(), x.max(axis=1))
        assert np.array_equal(t.argmin_axes([1]).to_numpy(), x.argmin(axis=1))


@pytest.mark.parametrize("dt", DTYPES[:3])
@pytest.mark.parametrize("rows,cols", [(63, 40000), (64, 40000), (65, 30001), (333, 20002), (1001, 130001), (4099, 640)])
def test_column_parts(dev, dt, rows, cols):
    rng = np.random.default_rng(rows)
    x = ints(rng, (rows, cols), dt)
    for t in (inside(dev, x, 1), mid(dev, x)):
        assert np.array_equal(t.sum_axes([0]).to_numpy(), x.sum(axis=0, dtype=x.dtype))
        assert np.array_equal(t.max_axes([0]).to_numpy(), x.max(axis=0))
        assert np.array_equal(t.argmin_axes([0]).to_numpy(), x.argmin(axis=0))


@pytest.mark.parametrize("rows,cols", [(40000, 63), (64, 40000)])
def test_nan(dev, rows, cols):
    """A NaN reaches the sum of its row or column and no other."""
    rng = np.random.default_rng(1)
    x = ints(rng, (rows, cols), np.float64)
    x[5, 7] = np.nan
    for axis in (0, 1):
        got = rt.asarray(x, device=dev).sum_axes([axis]).to_numpy()
        assert np.array_equal(got, x.sum(axis=axis), equal_nan=True)


@pytest.mark.parametrize("dt", DTYPES[:4])
@pytest.mark.parametrize("rows,cols", [(20001, 33), (9000, 40), (127, 16384), (129, 16383), (450, 16386), (1000, 5001)])
def test_column_parts_side_by_side(dev, dt, rows, cols):
    """Few outputs with many parts, one part, two to six in one block, and more than six."""
    rng = np.random.default_rng(rows + cols)
    x = ints(rng, (rows, cols), dt)
    for t in (inside(dev, x, 1), mid(dev, x)):
        assert np.array_equal(t.sum_axes([0]).to_numpy(), x.sum(axis=0, dtype=x.dtype))
        if np.dtype(dt).kind != "c":
            assert np.array_equal(t.argmax_axes([0]).to_numpy(), x.argmax(axis=0))
