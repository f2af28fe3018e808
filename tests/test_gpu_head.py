"""The pieces of a greedy LM head where they can go wrong: the register GEMV
(every K it is built for, one tile and more tiles than workgroups, partial
batches) and the wide argmax (short rows, rows at every alignment, the last
partial vector, NaN of either sign, signed zeros, infinities)."""
import numpy as np
import pytest

import oracle
from test_gpu_llm import _gemv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [256 * i for i in range(1, 14)])
def test_gemv_every_width(ctx, k):
    # 13 x 256 = 3328 keeps the LDS kernel; the others run from registers
    for n, batch in ((16, 1), (16, 16), (16 * 37, 5), (16 * 771, 3)):
        rng = np.random.default_rng(n + k + batch)
        q, s = oracle.quantize_e4m3_rows(rng.normal(0, 0.02, (n, k)).astype(np.float32))
        x16 = rng.normal(0, 1, (batch, k)).astype(np.float16)
        y = _gemv(ctx, x16.view(np.uint16), q, s, batch, k, n)
        wq, xf = oracle.e4m3_to_f32(q).astype(np.float64), x16.astype(np.float64)
        bound = 1e-5 * (np.abs(xf) @ np.abs(wq).T) * s + 1e-30  # as in test_gpu_llm.py
        assert np.all(np.abs(y - (xf @ wq.T) * s) <= bound), (n, batch)


def _first_of_largest(x):
    """By bits: NaN above everything, -0 below +0; the first of equals."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32)
    key = np.where(u >> 31, ~u, u | 0x80000000).astype(np.uint64)
    key[np.isnan(x)] = 1 << 32
    return np.argmax(key, axis=1).astype(np.int32)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 63, 1021, 4096, 4099, 32769, 50257])
def test_argmax_edges(ctx, n):
    rng = np.random.default_rng(n)
    x = rng.normal(0, 1, (24, n)).astype(np.float32)
    x[1] = -np.inf
    x[2] = 0.0
    x[2, : n // 2] = -0.0                       # +0 lies above -0
    x[3] = -0.0
    x[4, -1] = 50.0                             # the last value
    x[5, 0] = 50.0
    x[6, rng.integers(n)] = np.nan
    x[7, n // 2:] = -np.float32(np.nan)         # NaN of the other sign; the first one
    x[8] = np.nan
    x[9, [n // 3, n // 2, n - 1]] = 9.0         # ties
    x[10, n // 2] = np.inf
    x[11, [0, n - 1]] = np.inf
    x[12] = -1.0
    x[12, n - 1] = np.float32(-0.99999994)      # one step above
    x[13] = np.finfo(np.float32).tiny * 2.0 ** -10  # subnormals, all the same
    dx, di = ctx.upload(x), ctx.empty((24,), np.int32)
    ctx.argmax(dx, 24, n, di)
    ctx.sync()
    assert np.array_equal(di.to_host(), _first_of_largest(x))
    dx.free()
    di.free()
