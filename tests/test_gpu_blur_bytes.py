"""The byte-strip blur (1 to 4 channels, any width and alignment) where it can
go wrong: rows shorter than one 8-byte load, strips of 496 bytes that end just
before, at and after the row's end, bands of 4 and of 8 rows with remainders,
unaligned buffers, and nothing written outside the image. Bytes are exact."""
import numpy as np
import pytest

import oracle
import strict_amd
from tests.util import seeded_bytes

pytestmark = pytest.mark.gpu
NT = oracle.default_threads()


def _reference(img, w, h, c, mode, delta=0, all_channels=False):
    if delta:
        img = oracle.adjust_brightness(img, delta, c, all_channels=all_channels)
    blur = oracle.blur5_config if mode == strict_amd.BLUR_CONFIG else oracle.blur5_reference
    return blur(img, w, h, c, nthreads=NT if img.size > 1 << 20 else 1)


def _gpu(ctx, img, w, h, c, mode, delta=0, flags=0, offset=0):
    src = ctx.upload(np.concatenate([np.full(offset, 9, np.uint8), img]))
    out = ctx.upload(np.full(offset + img.size + 16, 0xA5, np.uint8))
    s, d = src.view(offset, img.size), out.view(offset, img.size)
    if delta:
        ctx.brightness_blur5(s, d, w, h, c, delta, flags, mode)
    else:
        ctx.box_blur5(s, d, w, h, c, mode)
    ctx.sync()
    host = out.to_host()
    src.free()
    out.free()
    assert np.all(host[:offset] == 0xA5) and np.all(host[offset + img.size:] == 0xA5)
    return host[offset:offset + img.size]


@pytest.mark.parametrize("mode", [strict_amd.BLUR_CONFIG, strict_amd.BLUR_REFERENCE])
@pytest.mark.parametrize("c", [1, 2, 3, 4])
def test_strip_and_band_edges(ctx, c, mode):
    widths = {1, 2, 3, 4, 5, 7, 8, 9, 13}
    for edge in (496, 504, 992, 1000):  # strips and the halo beyond them
        widths |= {edge // c + k for k in range(-3, 4)}
    for i, w in enumerate(sorted(x for x in widths if x > 0)):
        for h in (1, 2, 5, 9) if w > 20 else (1, 2, 3, 4, 6, 17):
            img = seeded_bytes(w * h * c, seed=w * 31 + h)
            got = _gpu(ctx, img, w, h, c, mode, offset=i % 5)
            assert np.array_equal(got, _reference(img, w, h, c, mode)), (w, h)


@pytest.mark.parametrize("mode", [strict_amd.BLUR_CONFIG, strict_amd.BLUR_REFERENCE])
@pytest.mark.parametrize("c,delta,flags", [(1, -40, 0), (3, 40, 0), (4, 40, 0), (4, -255, 1), (2, 255, 0)])
def test_fused_brightness(ctx, c, delta, flags, mode):
    for w, h, offset in ((5, 3, 0), (333, 37, 0), (333, 37, 3), (701, 11, 0)):
        img = seeded_bytes(w * h * c, seed=w + c)
        got = _gpu(ctx, img, w, h, c, mode, delta, flags, offset)
        assert np.array_equal(got, _reference(img, w, h, c, mode, delta, bool(flags))), (w, h, offset)


@pytest.mark.parametrize("w,h,c,mode", [(12301, 3843, 1, strict_amd.BLUR_REFERENCE),
                                        (4099, 3845, 3, strict_amd.BLUR_CONFIG),
                                        (1001, 999, 4, strict_amd.BLUR_CONFIG),
                                        (2236, 2236, 4, strict_amd.BLUR_CONFIG),
                                        (2240, 2236, 4, strict_amd.BLUR_CONFIG)])
def test_large_images(ctx, w, h, c, mode):
    # 8-row bands (the first two); either side of the RGBA streaming kernel
    img = seeded_bytes(w * h * c, seed=5)
    assert np.array_equal(_gpu(ctx, img, w, h, c, mode), _reference(img, w, h, c, mode))


@pytest.mark.parametrize("mode", [strict_amd.BLUR_CONFIG, strict_amd.BLUR_REFERENCE])
@pytest.mark.parametrize("c", [1, 2, 3, 4])
def test_narrow_tall_images(ctx, c, mode):
    # either side of the sizes where a thread takes one pixel
    for h in (32767, 32768, 32771):
        for w in sorted({1, 2, 11 // c, 12 // c, 15 // c, 16 // c, 17 // c}):
            img = seeded_bytes(w * h * c, seed=w * 31 + c)
            got = _gpu(ctx, img, w, h, c, mode, offset=w % 3)
            assert np.array_equal(got, _reference(img, w, h, c, mode)), (w, h)
            got = _gpu(ctx, img, w, h, c, mode, -40, w % 2)
            assert np.array_equal(got, _reference(img, w, h, c, mode, -40, w % 2 == 1)), (w, h)


@pytest.mark.parametrize("mode", [strict_amd.BLUR_CONFIG, strict_amd.BLUR_REFERENCE])
def test_tallest_image(ctx, mode):
    # 2^29 rows of one byte: a wave for each 8 rows is a grid of 2^32 threads. The ends
    # and the middle are those of short images (2 rows beyond their own edges)
    h, n = 1 << 29, 1 << 24
    part = seeded_bytes(n, seed=9)
    src, out = ctx.empty((h,), np.uint8), ctx.upload(np.zeros(h, np.uint8))
    for s in range(0, h, n):
        src.view(s, n).copy_from_host(part)
    ctx.box_blur5(src, out, 1, h, 1, mode)
    ctx.sync()
    ref = _reference(part, 1, n, 1, mode)
    assert np.array_equal(out.view(0, n - 2).to_host(), ref[:-2])
    assert np.array_equal(out.view(h - n + 2, n - 2).to_host(), ref[2:])
    joint = np.concatenate([part[-8:], part[:8]])
    for s in (n, h // 2, h - n):
        assert np.array_equal(out.view(s - 6, 12).to_host(), _reference(joint, 1, 16, 1, mode)[2:-2])
        assert np.array_equal(out.view(s + 2, n - 4).to_host(), ref[2:-2]) or s == h - n
    src.free()
    out.free()


@pytest.mark.parametrize("delta,flags", [(40, 0), (40, 1), (-40, 0), (-40, 1), (0, 0)])
def test_large_rgba_with_brightness(ctx, delta, flags):
    # the RGBA streaming kernel with a partial last strip (2244 = 9 x 240 + 84
    # pixels) and band (2237 = 139 x 16 + 13 rows), with and without alpha
    w, h = 2244, 2237
    img = seeded_bytes(w * h * 4, seed=delta + flags + 50)
    got = _gpu(ctx, img, w, h, 4, strict_amd.BLUR_CONFIG, delta, flags)
    assert np.array_equal(got, _reference(img, w, h, 4, strict_amd.BLUR_CONFIG, delta, bool(flags)))
