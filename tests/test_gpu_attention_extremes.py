"""Decode attention with infinities in the caches, and with queries whose values
lie far apart, against the oracle's fp64 attention: a score of -inf has no
weight, an infinite V under a positive weight is infinite, infinities of both
signs and a score of +inf are NaN."""
import numpy as np
import pytest

import oracle.llm as ollm
from test_gpu_attention_edges import _inputs, _run

pytestmark = pytest.mark.gpu

# one split and several; one tile per split and (64 rows of 8 KV heads) several
SHAPES = [(64, 4, 4, 2, 100), (128, 16, 8, 3, 127), (128, 16, 1, 2, 700), (64, 12, 12, 2, 1030),
          (128, 16, 8, 64, 1000)]


def _same(got, q, k, v, lens, scale):
    with np.errstate(invalid="ignore", over="ignore"):
        ref = ollm.attn_decode(q, k.astype(np.float32), v.astype(np.float32), lens, scale)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isinf(got), np.isinf(ref))
    assert np.array_equal(got[np.isinf(got)], ref[np.isinf(ref)])
    f = np.isfinite(ref)
    # (the bound of test_gpu_attention_edges.py)
    assert np.max(np.abs(got[f] - ref[f]), initial=0.0) <= 1e-5 * np.max(np.abs(ref[f]), initial=1e-30)


def _case(d, heads, kvh, batch, max_pos):
    lens = [max_pos - 7 * b % 50 for b in range(batch)]
    q, k, v, n = _inputs(d + heads, batch, heads, kvh, d, max_pos, lens)
    q[:, :, 3] = np.abs(q[:, :, 3]) + 0.1  # the sign of a score through key value 3
    return q, k, v, n, float(np.float32(1 / np.sqrt(d)))


@pytest.mark.parametrize("d,heads,kvh,batch,max_pos", SHAPES)
def test_a_key_of_minus_infinity_has_no_weight(ctx, d, heads, kvh, batch, max_pos):
    q, k, v, n, scale = _case(d, heads, kvh, batch, max_pos)
    k[:, :, [0, 5, 40, 64, 93], 3] = -np.inf
    k[1, :, 16:48, 3] = -np.inf  # all of a wave's share of a tile
    for b in range(batch):
        k[b, 0, n[b] - 1, 3] = -np.inf
    got = _run(ctx, q, k, v, n, scale)
    assert np.isfinite(got).all()
    _same(got, q, k, v, n, scale)


@pytest.mark.parametrize("d,heads,kvh,batch,max_pos", SHAPES)
def test_infinite_values(ctx, d, heads, kvh, batch, max_pos):
    q, k, v, n, scale = _case(d, heads, kvh, batch, max_pos)
    v[0, :, 17, 5] = np.inf
    v[0, 0, 30, 8] = -np.inf
    v[0, 0, 50, 9], v[0, 0, 90, 9] = np.inf, -np.inf  # NaN
    for b in range(1, batch):  # a row's last position
        v[b, :, n[b] - 1, b % d] = np.inf
    got = _run(ctx, q, k, v, n, scale)
    assert np.isinf(got).any() and np.isnan(got).any()
    _same(got, q, k, v, n, scale)


@pytest.mark.parametrize("d,heads,kvh,batch,max_pos", SHAPES[:4])
def test_infinite_scores_and_nan(ctx, d, heads, kvh, batch, max_pos):
    q, k, v, n, scale = _case(d, heads, kvh, batch, max_pos)
    k[0, :, 21, 3] = np.inf
    k[1, 0, 3, 4] = np.nan
    got = _run(ctx, q, k, v, n, scale)
    assert np.isnan(got[0]).all() and np.isnan(got[1]).any()
    _same(got, q, k, v, n, scale)


@pytest.mark.parametrize("d", [64, 128])
def test_small_query_values_beside_a_large_one(ctx, d):
    # 2^10 on a key value of about 2^-12, 2^-6 on keys of about 16. Kept to
    # 2^-37 of the largest, the small ones are off by 2^-27 each: 2^-27 x 16 x
    # sqrt(d) is 1.4e-6 of a score, beside fp32 sums of d terms of 0.25 (up to
    # 2e-6): 2e-5 of the output holds four times both. Kept to 2^-25 of the
    # largest they would be off by 5e-3.
    q, k, v, n = _inputs(d, 3, 8, 4, d, 300, [300, 299, 130])
    q *= np.float32(2.0 ** -6)
    q[:, :, 7] = 2.0 ** 10
    k *= np.float16(16)
    k[..., 7] = (np.random.default_rng(1).normal(0, 2.0 ** -12, k.shape[:-1])).astype(np.float16)
    got = _run(ctx, q, k, v, n, 1.0)
    ref = ollm.attn_decode(q, k.astype(np.float32), v.astype(np.float32), n, 1.0)
    assert np.max(np.abs(got - ref)) <= 2e-5 * np.max(np.abs(ref))
