"""The elementwise pieces past the sizes where a grid of one thread per few values
would need 2^32 threads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op", ["gelu", "swiglu"])
def test_more_values_than_a_grid_has_threads_for(ctx, op):
    # in place over 2^35 + 8,003 values (128 GiB): the ends and the values around
    # the 2^32-nd thread are those of a short call on the same values
    n = 2 ** 35 + 8_003
    try:
        x = ctx.empty((n,), np.float32)
    except Exception:
        pytest.skip("no device memory for 128 GiB")
    ctx.fill(0.0, x, n)
    part = np.random.default_rng(0).normal(0, 2, 3000).astype(np.float32)
    small = ctx.upload(part)
    starts = (0, 2 ** 34 - 1500, 2 ** 35 - 1500, n - 3000)
    for s in starts:
        ctx.saxpy(0.0, small, small, x.ptr + 4 * s, 3000)

    def run(buf, count):
        if op == "gelu":
            ctx.gelu(buf, buf, count)
        else:
            ctx.swiglu(buf, buf, buf, count)

    run(small, 3000)
    run(x, n)
    ctx.sync()
    ref = small.to_host()
    assert np.abs(ref).max() > 1
    got = ctx.empty((3000,), np.float32)
    for s in starts:
        ctx.saxpy(0.0, x.ptr + 4 * s, x.ptr + 4 * s, got, 3000)
        ctx.sync()
        assert np.array_equal(got.to_host(), ref), s
    for b in (x, small, got):
        b.free()
