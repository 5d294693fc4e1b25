"""Tensors past 2^31 elements (a 16 GiB f64 array): a contiguous elementwise op whose merged axis
holds 2^31 + 2^21 elements, reductions over a reduced extent of that size (factored into two
reduced dims) and a reduction producing that many outputs (processed in pieces of the kept axis).
DeviceFaer has no such limit, so neither may the device."""
import math

import numpy as np
import pytest

import rstsr_amd as rt

pytestmark = pytest.mark.gpu

ROWS, COLS = 1 << 21, 1025  # 2,149,580,800 elements > 2^31


@pytest.fixture(scope="module")
def big(dev):
    rng = np.random.default_rng(20261260)
    v = rng.normal(size=COLS)
    tv = rt.asarray(v, device=dev)
    a = tv.broadcast_to([ROWS, COLS]).to_contig()  # c-contiguous 16 GiB
    return v, tv, a


def test_elementwise_past_2_31(dev, big):
    v, tv, a = big
    flat = a.reshape([ROWS * COLS])
    assert flat.shape == (ROWS * COLS,) and ROWS * COLS > 2 ** 31
    c = flat + flat  # one merged axis of 2^31 + 2^21 elements
    c2 = c.reshape([ROWS, COLS])
    for r in (0, ROWS // 2, ROWS - 1):
        assert np.array_equal(c2[r].to_numpy(), 2 * v)
    e = c2 - (tv + tv)  # broadcast row: every element must be exactly zero
    assert np.all(e.max_axes([1]).to_numpy() == 0) and np.all(e.min_axes([1]).to_numpy() == 0)


def test_reduction_over_2_31_elements(dev, big):
    v, tv, a = big
    flat = a.reshape([ROWS * COLS])
    s = flat.sum_axes([0]).to_scalar()
    exact = ROWS * math.fsum(v.tolist())  # a power-of-two multiple: exact
    assert abs(s - exact) <= 4 * 2.0 ** -53 * abs(exact) + 1e-300
    assert flat.argmax_all() == int(np.argmax(v))
    assert flat.max_all() == float(np.max(v))
    # a reversed view starts with v reversed: its first minimum is argmin(v[::-1])
    assert flat[::-1].argmin_all() == int(np.argmin(v[::-1]))


def test_reduction_with_2_31_outputs(dev, big):
    v, tv, a = big
    col = a.reshape([ROWS * COLS, 1])
    out = col.sum_axes([1])  # 2^31 + 2^21 outputs, one element each
    assert out.shape == (ROWS * COLS,)
    e = out.reshape([ROWS, COLS]) - a
    assert np.all(e.max_axes([1]).to_numpy() == 0) and np.all(e.min_axes([1]).to_numpy() == 0)


def test_solve_with_2_27_columns(dev):
    """33 rows x (2^27 + 3) right-hand sides of a diagonal solve, more than one launch covers."""
    import ctypes as C

    from rstsr_amd import abi

    s, r = 33, (1 << 27) + 3
    a = rt.asarray(np.diag(np.full(s, 2.0, dtype=np.float32)), device=dev)
    b = rt.full((s, r), 6.0, dtype=np.float32, device=dev)
    one = np.array(1, dtype=np.float32)
    abi.check(abi.lib().rstsr_hip_driver_trsm(C.c_void_p(dev._ctx_ptr()), rt._code(np.float32), 0, 101, 141, 122, 111, 131,
                                              s, r, one.ctypes.data, a.as_ptr(), s, b.as_ptr(), r))
    assert b.max_all() == 3.0 and b.min_all() == 3.0


def test_product_with_2_34_outputs(dev):
    """An f64 outer product of 128 GiB, whose smallest tiles would need more threads than a launch
    holds: the tuner leaves those out."""
    n = 1 << 17
    x = np.arange(n, dtype=np.float64)
    rt.empty_cache(dev)
    a, b = rt.asarray(x.reshape(n, 1), device=dev), rt.asarray(x.reshape(1, n), device=dev)
    try:
        c = a % b
    except rt.RSTSRError as e:
        if e.args[0] != "MemoryError":
            raise
        pytest.skip("no 128 GiB for the output")
    for i in (0, 1, n // 2 + 1, n - 1):
        assert np.array_equal(c[i].to_numpy(), i * x)
        assert np.array_equal(c[:, i].to_contig().to_numpy(), i * x)
    del c
    rt.empty_cache(dev)


def test_matrix_vector_product_with_2_28_rows(dev):
    """[2^28 + 5, 1] @ [1], row by row and (a vector of the matrix's rows) as columns: more rows than
    one launch covers."""
    m = (1 << 28) + 5
    a = rt.full((m, 1), 3.0, dtype=np.float32, device=dev)
    x = rt.asarray(np.array([7.0], dtype=np.float32), device=dev)
    for mat in (a, a.reshape([1, m]).transpose()):
        y = mat % x
        assert y.shape == (m,) and y.max_all() == 21.0 and y.min_all() == 21.0


def test_reductions_with_many_outputs(dev):
    """2^26 + 1 rows of 512 (a wave per row would be 2^32 threads), and 46341^2 > 2^31 outputs none of
    whose axes is long."""
    row = np.arange(512, dtype=np.float32)
    rows = (1 << 26) + 1
    t = rt.asarray(row.reshape(1, 512), device=dev).broadcast_to([rows, 512])
    s = t.sum_axes([1])
    assert s.shape == (rows,) and s.max_all() == row.sum() and s.min_all() == row.sum()
    n = 46341
    pairs = np.arange(2 * n, dtype=np.float32).reshape(1, n, 2)
    s = rt.asarray(pairs, device=dev).broadcast_to([n, n, 2]).sum_axes([2])
    e = s - rt.asarray(pairs.sum(axis=2), device=dev)
    assert s.shape == (n, n) and e.max_all() == 0 and e.min_all() == 0


def test_integer_product_with_2_32_outputs(dev):
    """An i32 outer product of 2^32 + 2^16 outputs, a thread each."""
    m, n = (1 << 16) + 1, 1 << 16
    a = rt.asarray(np.arange(m, dtype=np.int32).reshape(m, 1), device=dev)
    b = rt.asarray((np.arange(n, dtype=np.int32) % 1000).reshape(1, n), device=dev)
    c = a % b
    for i in (0, 1, m // 2, m - 1):
        assert np.array_equal(c[i].to_numpy(), i * (np.arange(n, dtype=np.int32) % 1000))
