"""Element-wise passes at the edges of their packs and tiles.

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


# rows x columns of at least 4096 elements: rows shorter than a pack, one off a pack, one off the
# elements of a block and of a thread's packs
FLAT = [(4099, 1), (2048, 2), (1401, 3), (1024, 4), (821, 5), (257, 17), (64, 64), (7, 1023), (3, 4097), (1, 70001)]


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("shape", FLAT)
def test_flat_broadcast_forms(dev, dt, shape):
    rng = np.random.default_rng(shape[0])
    r, c = shape
    forms = [(r, c), (r, 1), (1, c), (1, 1)]
    for lead_a, lead_b in ((0, 0), (1, 3)):
        a = ints(rng, (r, c), dt)
        ta = inside(dev, a, lead_a)
        for f in forms:
            b = ints(rng, f, dt)
            tb = inside(dev, b, lead_b)
            assert np.array_equal((ta - tb).to_numpy(), a - b), (f, lead_a, lead_b)
            assert np.array_equal((tb - ta).to_numpy(), b - a), (f, lead_a, lead_b)
        # in place, at an offset: nothing beside the view changes
        buf = np.full(a.size + 9, FILL, dtype=dt)
        out = rt.asarray(buf, device=dev)
        v = out._view(([r, c], [c, 1], lead_a))
        v.assign(ta)
        want = buf.copy()
        want[lead_a:lead_a + a.size] = a.reshape(-1)
        assert np.array_equal(out.to_numpy(), want)
        # a strided operand beside a contiguous one
        assert np.array_equal((ta + mid(dev, a)).to_numpy(), a + a)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("shape", [(5, 33, 65), (63, 31, 64), (2, 129, 66), (64, 64, 64), (3, 7, 1000), (1, 4097, 3)])
def test_tiled_edges(dev, dt, shape):
    rng = np.random.default_rng(7)
    x = ints(rng, shape, dt)
    t = mid(dev, x)
    c = rt.asarray(x, device=dev)
    for p in ((2, 1, 0), (2, 0, 1), (1, 2, 0), (1, 0, 2), (0, 2, 1)):
        xp = x.transpose(p)
        b = ints(rng, (1,) + xp.shape[1:], dt)
        for u in (t, c):
            up = u.transpose(list(p))
            assert np.array_equal(up.to_contig().to_numpy(), xp), p
            assert np.array_equal((up + inside(dev, b, 1)).to_numpy(), xp + b), p
            assert np.array_equal((up + u.transpose(list(p))).to_numpy(), xp + xp), p
