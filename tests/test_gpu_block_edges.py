"""RMSNorm, LayerNorm, RoPE, SwiGLU and GELU where their kernels can go wrong:
rows around every register variant's length and off the vectors of 4, few rows,
unaligned and in-place buffers, head counts that leave a partial unit, head
dimensions of 2 to 512, and angles over the whole range of positions.
Tolerances are those of test_gpu_ops.py (1 ulp; 8 for SwiGLU's expf and divide)."""
import numpy as np
import pytest

import oracle.llm as ollm
from test_gpu_ops import _ulps

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 3, 4, 5, 63, 255, 257, 768, 1000, 1023, 1024, 1025, 2047, 2048, 2049, 8191, 8192, 8193,
           20001]


def _at(ctx, x, offset):
    """x on the device, `offset` values into its buffer."""
    buf = ctx.upload(np.concatenate([np.full(offset, np.nan, np.float32), x.ravel(),
                                     np.full(8, np.nan, np.float32)]))
    return buf, buf.view(4 * offset, x.nbytes, np.float32, x.shape)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("rows", [1, 3, 6])
def test_norm_lengths(ctx, rows, offset):
    for n in LENGTHS:
        rng = np.random.default_rng(n + rows)
        x = (rng.normal(0, 2, (rows, n)) + 1).astype(np.float32)
        g = (1 + rng.normal(0, 0.2, n)).astype(np.float32)
        b = rng.normal(0, 0.3, n).astype(np.float32)
        eps = float(np.float32(1e-5))
        bufs = [_at(ctx, a, offset) for a in (x, g, b)]
        (_, dx), (_, dg), (_, db) = bufs
        out, dy = _at(ctx, np.zeros_like(x), offset)
        ctx.layernorm(dx, dg, db, dy, rows, n, eps)
        ctx.sync()
        assert _ulps(dy.to_host(), ollm.layer_norm(x, g, b, eps)).max() <= 1, n
        ctx.rmsnorm(dx, dg, dx, rows, n, eps)  # in place
        ctx.sync()
        assert _ulps(dx.to_host(), ollm.rms_norm(x, g, eps)).max() <= 1, n
        for buf in [bufs[0][0], out]:  # nothing past the rows was written
            assert np.all(np.isnan(buf.to_host()[offset + rows * n:]))
        for buf, _ in bufs + [(out, None)]:
            buf.free()


@pytest.mark.parametrize("heads,d,theta", [(1, 2, 1e4), (3, 6, 1e4), (5, 64, 1e6), (4, 130, 500.0),
                                           (9, 256, 1e4), (2, 386, 1e6), (6, 512, 0.5)])
def test_rope_shapes_and_positions(ctx, heads, d, theta):
    positions = np.array([0, 1, -1, 2, 1023, -70000, 1_000_003, 2**31 - 1, -2**31], np.int32)
    rng = np.random.default_rng(d)
    x = rng.normal(0, 1, (positions.size, heads, d)).astype(np.float32)
    dx, dp = ctx.upload(x), ctx.upload(positions)
    ctx.rope(dx, dp, positions.size, heads, d, theta)
    ctx.sync()
    cos, sin = ollm.rope_tables(ollm.inv_freq(theta, d), positions)
    assert _ulps(dx.to_host(), ollm.rope(x, cos, sin)).max() <= 1
    dx.free()
    dp.free()


@pytest.mark.parametrize("offset", [0, 1])
def test_elementwise_lengths(ctx, offset):
    for n in (1, 2, 3, 4, 5, 9, 1023, 2047, 2048, 2049, 4099, 100_001):
        rng = np.random.default_rng(n)
        gate, up = rng.normal(0, 4, n).astype(np.float32), rng.normal(0, 2, n).astype(np.float32)
        (bg, dg), (bu, du), (bo, do) = (_at(ctx, a, offset) for a in (gate, up, np.zeros_like(gate)))
        ctx.swiglu(dg, du, do, n)
        ctx.sync()
        assert _ulps(do.to_host(), ollm.silu(gate) * up).max() <= 8, n
        ctx.gelu(dg, dg, n)  # in place
        ctx.sync()
        err = np.abs(dg.to_host().astype(np.float64) - ollm.gelu_tanh(gate))
        assert np.all(err <= 4 * 2.0 ** -23 * np.abs(gate.astype(np.float64)) + 1e-30), n
        for buf in (bg, bo):
            assert np.all(np.isnan(buf.to_host()[offset + n:]))
        for buf in (bg, bu, bo):
            buf.free()
