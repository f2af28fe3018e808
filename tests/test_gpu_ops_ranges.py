"""The elementwise pieces past the sizes where a grid of one thread per few values
would need 2^32 threads, and RoPE at the ends of theta."""
import numpy as np
import pytest

import oracle.llm as ollm

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


@pytest.mark.parametrize("theta", [np.inf, 3e38, 1.0, 1e-3])
def test_rope_at_the_ends_of_theta(ctx, theta):
    # an infinite theta turns the first pair by the position and leaves the others
    rows, heads, d = 9, 3, 64
    rng = np.random.default_rng(4)
    x = rng.normal(0, 1, (rows, heads, d)).astype(np.float32)
    positions = np.arange(rows, dtype=np.int32)
    freq = np.array([float(np.float32(theta)) ** (-2.0 * i / d) for i in range(d // 2)]).astype(np.float32)
    assert freq[0] == 1.0
    dx, dp = ctx.upload(x), ctx.upload(positions)
    ctx.rope(dx, dp, rows, heads, d, float(theta))
    ctx.sync()
    cos, sin = ollm.rope_tables(freq, positions)
    ref = ollm.rope(x, cos, sin)
    # one rounding per product and sum, and of cos and sin
    assert np.max(np.abs(dx.to_host() - ref)) <= 4 * 2.0 ** -23 * np.max(np.abs(ref))
    for b in (dx, dp):
        b.free()
