"""Decode attention where its kernels can go wrong: lengths at the edges of the
16-position blocks, of a wave's share and of the 128- / 256-position tiles, one
split (no merge) and many, several tiles per split, every group size class,
unused columns, NaN in the cache past a row's length, very large and very
small queries, and a softmax that one key dominates.

Bound: the oracle's attention is fp64; scores, exponentials and sums here are
fp32 or better. A score s has an error of about d x 2^-24 x sum |q k|, at most
2e-6 at these sizes (|s| up to ~6), which moves a weight by as much, relatively;
1e-5 of the largest output holds several times that."""
import numpy as np
import pytest

import oracle.llm as ollm

pytestmark = pytest.mark.gpu


def _run(ctx, q, k, v, lens, scale):
    batch, heads, d = q.shape
    kvh, max_pos = k.shape[1], k.shape[2]
    bufs = [ctx.upload(a) for a in (q, k.view(np.uint16), v.view(np.uint16), lens)]
    out = ctx.upload(np.full((batch, heads, d), np.nan, np.float32))
    ctx.attn_decode(*bufs, out, batch, heads, kvh, d, max_pos, scale)
    ctx.sync()
    got = out.to_host()
    for b in bufs + [out]:
        b.free()
    return got


def _inputs(seed, batch, heads, kvh, d, max_pos, lens):
    rng = np.random.default_rng(seed)
    q = rng.normal(0, 1, (batch, heads, d)).astype(np.float32)
    k = rng.normal(0, 1, (batch, kvh, max_pos, d)).astype(np.float16)
    v = rng.normal(0, 1, (batch, kvh, max_pos, d)).astype(np.float16)
    return q, k, v, np.array(lens, np.int32)


def _check(got, q, k, v, lens, scale):
    ref = ollm.attn_decode(q, k.astype(np.float32), v.astype(np.float32), lens, scale)
    assert np.max(np.abs(got - ref)) <= 1e-5 * max(np.max(np.abs(ref)), 1e-30)


@pytest.mark.parametrize("heads,kvh", [(1, 1), (4, 4), (4, 2), (3, 1), (10, 2), (8, 1), (16, 1)])
@pytest.mark.parametrize("d", [64, 128])
def test_lengths_at_tile_edges(ctx, d, heads, kvh):
    lens = [-3, 0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 300, 999]
    for max_pos in (300, 127):  # several splits (300 is no multiple of 16); one split
        q, k, v, n = _inputs(d + heads, len(lens), heads, kvh, d, max_pos, lens)
        for b, L in enumerate(lens):  # what lies past a row's length does not matter
            k[b, :, max(0, L):] = np.nan
            v[b, :, max(0, L):] = np.nan
        got = _run(ctx, q, k, v, n, 1 / np.sqrt(d))
        _check(got, q, np.nan_to_num(k), np.nan_to_num(v), n, 1 / np.sqrt(d))
        assert not got[:2].any()


@pytest.mark.parametrize("d,heads,kvh,batch,max_pos", [(128, 16, 8, 64, 1000), (64, 12, 12, 48, 1030)])
def test_several_tiles_per_split(ctx, d, heads, kvh, batch, max_pos):
    lens = np.random.default_rng(1).integers(1, max_pos + 1, batch)
    q, k, v, n = _inputs(2, batch, heads, kvh, d, max_pos, lens)
    _check(_run(ctx, q, k, v, n, 1 / np.sqrt(d)), q, k, v, n, 1 / np.sqrt(d))


@pytest.mark.parametrize("factor", [1e-30, 1e-6, 3e4, 1e30])
def test_query_ranges(ctx, factor):
    # the scale brings the scores back to order 1; each head has its own range
    q, k, v, n = _inputs(3, 2, 4, 2, 128, 400, [400, 77])
    q = (q * np.float32(factor)).astype(np.float32)
    q[:, 1] *= np.float32(2.0 ** -9)
    scale = float(np.float32(1 / np.sqrt(128) / factor))
    _check(_run(ctx, q, k, v, n, scale), q, k, v, n, scale)


def test_one_key_dominates(ctx):
    q, k, v, n = _inputs(4, 2, 16, 8, 128, 700, [700, 130])
    k[:, :, 129] = 6.0 * np.sign(q.reshape(2, 8, 2, 128)[:, :, 0]).astype(np.float16)
    _check(_run(ctx, q, k, v, n, 1.0), q, k, v, n, 1.0)


# Calls whose splits of one tile would need over SH_ATTN_NOALLOC_MAX_BYTES of
# partials or more than 1,024 splits: one split of 192 positions (a tile and a
# half); 6 splits of 448; one of 192 (less than a tile of 256); 410 of 320
@pytest.mark.parametrize("d,heads,kvh,batch,max_pos,lo", [(128, 16, 1, 2048, 130, 65), (128, 16, 1, 97, 2600, 1),
                                                          (64, 16, 1, 4000, 130, 1), (128, 4, 1, 1, 131200, 131200)])
def test_splits_that_are_no_multiple_of_a_tile(ctx, d, heads, kvh, batch, max_pos, lo):
    tile = 128 if d == 128 else 256
    tiles = -(-max_pos // tile)
    fine = -(-tiles // max(1, -(-tiles * batch * kvh // 2048)))
    assert fine > 1024 or batch * heads * fine * (d + 2) * 4 > 16 << 20
    lens = np.random.default_rng(1).integers(lo, max_pos + 1, batch)
    lens[0] = max_pos
    q, k, v, n = _inputs(6, batch, heads, kvh, d, max_pos, lens)
    _check(_run(ctx, q, k, v, n, 1 / np.sqrt(d)), q, k, v, n, 1 / np.sqrt(d))
