"""Decode attention under graph capture: once a context has its work buffer, calls
of other shapes up to SH_ATTN_NOALLOC_MAX_BYTES of partials do not allocate."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

THREAD_LOCAL = 1  # hipStreamCaptureModeThreadLocal


@pytest.fixture(scope="module")
def hip():
    return ctypes.CDLL("libamdhip64.so")


@pytest.mark.parametrize("batch,heads,kv_heads,d,positions", [(4, 24, 8, 128, 4096), (8, 64, 16, 64, 8192)])
def test_finer_splits_in_a_captured_call(hip, batch, heads, kv_heads, d, positions):
    import strict_amd
    with strict_amd.Context(0) as ctx:
        rng = np.random.default_rng(3)
        q = ctx.upload(rng.normal(0, 1, (batch, heads, d)).astype(np.float32))
        kv = [ctx.upload(rng.normal(0, 1, (batch, kv_heads, positions, d)).astype(np.float16)) for _ in range(2)]
        lengths = ctx.upload(np.full(batch, positions, np.int32))
        out = ctx.empty((batch, heads, d), np.float32)
        ctx.attn_decode(q, *kv, lengths, out, 1, 1, 1, d, 16, 0.1)  # the work buffer
        ctx.sync()
        stream = ctypes.c_void_p(ctx.stream())
        graph, run = ctypes.c_void_p(), ctypes.c_void_p()
        assert hip.hipStreamBeginCapture(stream, THREAD_LOCAL) == 0
        try:
            ctx.attn_decode(q, *kv, lengths, out, batch, heads, kv_heads, d, positions, 0.1)
        finally:
            ended = hip.hipStreamEndCapture(stream, ctypes.byref(graph))
        assert ended == 0
        assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
        for i in range(3):
            q.copy_from_host(rng.normal(0, 1, (batch, heads, d)).astype(np.float32))
            ctx.sync()
            assert hip.hipGraphLaunch(run, stream) == 0
            ctx.sync()
            got = out.to_host()
            ctx.fill(0.0, out, batch * heads * d)
            ctx.attn_decode(q, *kv, lengths, out, batch, heads, kv_heads, d, positions, 0.1)
            ctx.sync()
            assert np.array_equal(got, out.to_host()) and np.abs(got).max() > 0, i
        assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
        for b in (q, *kv, lengths, out):
            b.free()
