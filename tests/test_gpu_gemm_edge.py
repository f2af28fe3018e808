"""The any-shape GEMM kernel behind sh_gemm_bf16 and sh_gemm_fp8 where it can
go wrong: remainders of its 64- and 128-wide tiles, of its 64-element (bf16) and
128-element (fp8) K stages and of its 16-byte loads, operands shorter than one
load, odd leading dimensions, unaligned operands, both tile sizes and the
four-group variant, rows and columns past the matrix that hold NaN.

Bound: the result's bf16 rounding (7 stored bits: at most 2^-8 of the value)
plus fp32 sums of exact products, K x 2^-24 of the sum of their magnitudes."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 1, 1), (1, 3, 2), (2, 1, 7), (3, 2, 5), (1, 300, 1), (16, 16, 8), (17, 9, 33),  # tiny spans
    (63, 65, 63), (64, 64, 64), (65, 63, 129), (130, 70, 127), (100, 37, 50),
    (128, 128, 257), (33, 1003, 517), (200, 5, 1000),
    (70, 66, 512), (64, 130, 1029), (16, 257, 1555),  # four groups
    (1921, 2047, 65), (2500, 3001, 40),               # 128 x 128 tiles (bf16; both)
    (256, 512, 128), (512, 768, 320),                 # multiples of 256, too few tiles for those
]


def _place(ctx, x, ld, offset, fill):
    """x [r, c] on the device with leading dimension ld, `offset` elements into
    its buffer, everything around it `fill`."""
    r, c = x.shape
    host = np.full(offset + r * ld + 64, fill, x.dtype)
    for i in range(r):
        host[offset + i * ld: offset + i * ld + c] = x[i]
    buf = ctx.upload(host)
    size = ((r - 1) * ld + c) * x.itemsize
    return buf, buf.view(offset * x.itemsize, size, x.dtype, (size // x.itemsize,))


def _c(ctx, m, n, ldc, offset):
    mark = np.full(offset + m * ldc + 64, 0x1234, np.uint16)
    buf = ctx.upload(mark)
    return buf, buf.view(offset * 2, ((m - 1) * ldc + n) * 2, np.uint16)


def _result(buf, m, n, ldc, offset):
    """C, after checking that nothing outside it was written."""
    host = buf.to_host()
    outside = np.ones(host.size, bool)
    for i in range(m):
        outside[offset + i * ldc: offset + i * ldc + n] = False
    assert np.all(host[outside] == 0x1234)
    return np.stack([host[offset + i * ldc: offset + i * ldc + n] for i in range(m)])


def _check(c_bits, a, b):
    ref = a.astype(np.float64) @ b.astype(np.float64)
    terms = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    bound = 2.0 ** -8 * np.abs(ref) + a.shape[1] * 2.0 ** -24 * terms + 1e-38
    assert np.all(np.abs(oracle.bf16_to_f32(c_bits) - ref) <= bound)


# pad: extra elements of each leading dimension; offset: elements before the operand
@pytest.mark.parametrize("pad,offset", [(0, 0), (3, 1), (8, 8)])
def test_bf16_edges(ctx, pad, offset):
    nan = np.uint16(0x7FC0)
    for m, n, k in SHAPES:
        rng = np.random.default_rng(m * 31 + n * 7 + k)
        a = oracle.f32_to_bf16(rng.normal(0, 1, (m, k)).astype(np.float32))
        b = oracle.f32_to_bf16(rng.normal(0, 1, (k, n)).astype(np.float32))
        ba, va = _place(ctx, a, k + pad, offset, nan)
        bb, vb = _place(ctx, b, n + pad, offset, nan)
        bc, vc = _c(ctx, m, n, n + pad, offset)
        ctx.gemm_bf16(va, vb, vc, m, n, k, k + pad, n + pad, n + pad)
        ctx.sync()
        _check(_result(bc, m, n, n + pad, offset), oracle.bf16_to_f32(a), oracle.bf16_to_f32(b))
        for x in (ba, bb, bc):
            x.free()


@pytest.mark.parametrize("pad,offset", [(0, 0), (3, 1), (16, 16)])
def test_fp8_edges(ctx, pad, offset):
    nan = np.uint8(0x7F)
    for m, n, k in SHAPES:
        rng = np.random.default_rng(m * 31 + n * 7 + k)
        a, sa = oracle.quantize_e4m3_rows(rng.normal(0, 1, (m, k)).astype(np.float32))
        b, sb = oracle.quantize_e4m3_rows(rng.normal(0, 1, (n, k)).astype(np.float32))
        ba, va = _place(ctx, a, k + pad, offset, nan)
        bb, vb = _place(ctx, b, k + pad, offset, nan)
        bc, vc = _c(ctx, m, n, n + pad, offset)
        dsa, dsb = ctx.upload(sa), ctx.upload(sb)
        ctx.gemm_fp8(va, dsa, vb, dsb, vc, m, n, k, k + pad, k + pad, n + pad)
        ctx.sync()
        _check(_result(bc, m, n, n + pad, offset), oracle.e4m3_to_f32(a) * sa[:, None],
               (oracle.e4m3_to_f32(b) * sb[:, None]).T)
        for x in (ba, bb, bc, dsa, dsb):
            x.free()


@pytest.mark.parametrize("m,n,k", [(65, 67, 129), (30, 130, 1029)])
def test_bf16_special_values_stay_in_their_row_and_column(ctx, m, n, k):
    # an infinity in A reaches its row, a NaN in B its column, and no other;
    # subnormal operands count as what they are
    rng = np.random.default_rng(k)
    a = rng.normal(0, 1, (m, k)).astype(np.float32)
    b = rng.normal(0, 1, (k, n)).astype(np.float32)
    a[7, k - 1] = np.inf
    b[k - 1, 11] = np.nan
    a[9, :] = 2.0 ** -130
    a16, b16 = oracle.f32_to_bf16(a), oracle.f32_to_bf16(b)
    da, db, dc = ctx.upload(a16), ctx.upload(b16), ctx.empty((m, n), np.uint16)
    ctx.gemm_bf16(da, db, dc, m, n, k)
    ctx.sync()
    c = oracle.bf16_to_f32(dc.to_host())
    with np.errstate(invalid="ignore"):
        ref = oracle.bf16_to_f32(a16).astype(np.float64) @ oracle.bf16_to_f32(b16).astype(np.float64)
    assert np.array_equal(np.isnan(c), np.isnan(ref)) and np.array_equal(np.isinf(c), np.isinf(ref))
    fine = np.isfinite(ref)
    assert np.allclose(c[fine], ref[fine], rtol=2.0 ** -8, atol=1e-3)
    row = fine[9]
    print("subnormal row: max rel err", np.max(np.abs(c[9][row] - ref[9][row])) / np.max(np.abs(ref[9][row])))
    for x in (da, db, dc):
        x.free()
