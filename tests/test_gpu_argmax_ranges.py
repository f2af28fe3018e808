"""argmax at the ends of its ranges: rows of nearly 2^31 values (32-bit sums of
an index and a stride wrap there), more rows than a grid of 1,024 threads each
can have, and rows at the lengths where the kernels change."""
import numpy as np
import pytest

from test_gpu_head import _first_of_largest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2 ** 31 - 1, 2 ** 31 - 131_070, 2 ** 31 - 40_003])
def test_argmax_of_the_longest_rows(ctx, n):
    x, i = ctx.empty((n,), np.float32), ctx.empty((1,), np.int32)
    ctx.fill(-2.0, x, n)

    def put(at, value):
        one = ctx.upload(np.array([value], np.float32))
        ctx.saxpy(1.0, one, one, x.ptr + 4 * at, 1)  # value + value
        ctx.sync()
        one.free()

    def found():
        ctx.argmax(x, 1, n, i)
        ctx.sync()
        return int(i.to_host()[0])

    assert found() == 0
    for at in (n - 1, n - 5, 2 ** 30, 3):  # each larger than the last
        put(at, 1.0 + (n - at) * 2.0 ** -31)
        assert found() == at
    put(n - 2, np.nan)
    assert found() == n - 2
    x.free()
    i.free()


@pytest.mark.parametrize("rows,n", [(5_000_000, 4), (4_200_000, 1030)])
def test_argmax_of_many_rows(ctx, rows, n):
    rng = np.random.default_rng(n)
    part = rng.normal(0, 1, (1000, n)).astype(np.float32)
    part[7, n // 2] = np.nan
    dx, di = ctx.empty((rows * n,), np.float32), ctx.empty((rows,), np.int32)
    ctx.fill(0.0, dx, rows * n)
    first, last = ctx.upload(part), ctx.upload(part[::-1].copy())
    ctx.saxpy(0.0, first, first, dx.ptr, 1000 * n)
    ctx.saxpy(0.0, last, last, dx.ptr + 4 * (rows - 1000) * n, 1000 * n)
    ctx.argmax(dx, rows, n, di)
    ctx.sync()
    got, ref = di.to_host(), _first_of_largest(part)
    assert np.array_equal(got[:1000], ref) and np.array_equal(got[-1000:], ref[::-1])
    assert not got[1000:-1000].any()
    for b in (dx, di, first, last):
        b.free()


@pytest.mark.parametrize("n", [1, 64, 65, 255, 257, 1023, 1024, 1025, 8191, 8192, 8193, 8196])
def test_argmax_where_the_kernels_change(ctx, n):
    rng = np.random.default_rng(n)
    x = rng.integers(-3, 4, (37, n)).astype(np.float32)  # many ties
    x[1] = -np.inf
    x[2] = np.nan
    x[3, rng.integers(n)] = -np.float32(np.nan)
    x[4], x[4, n // 2] = -0.0, 0.0
    x[5, n - 1] = 9.0
    dx, di = ctx.upload(x), ctx.empty((37,), np.int32)
    ctx.argmax(dx, 37, n, di)
    ctx.sync()
    assert np.array_equal(di.to_host(), _first_of_largest(x))
    dx.free()
    di.free()
