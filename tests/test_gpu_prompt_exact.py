"""sh_llm_generate's one-pass prompt leaves what steps over the same tokens
leave, bit for bit: KV caches of every layer, lengths, history, and the logits
and token of the step that follows. The pass sums in the step kernels' own
order, so there is no tolerance."""
import numpy as np
import pytest

from strict_amd import llm
from test_gpu_llm import GPT2_SMALL_TEST, QWEN_SMALL, _randomize_small_params
from test_gpu_prefill import _state, _stepwise

pytestmark = pytest.mark.gpu

QWEN_WIDE = llm.QWEN3_0_6B.with_(layers=3, vocab=512, max_batch=16)
GPT2_WIDE = llm.GPT2_SMALL.with_(layers=3, vocab=512, max_batch=16)


def _model(ctx, cfg, std=0.02):
    m = llm.Model(ctx, cfg)
    m.init_random(seed=7, stddev=std)
    _randomize_small_params(m, 1)
    return m


def _same(got, ref, what):
    (gc, gl, glen, gh), (rc, rl, rlen, rh) = got, ref
    assert np.array_equal(glen, rlen) and np.array_equal(gh, rh), what
    for i, (g, r) in enumerate(zip(gc, rc)):
        assert np.array_equal(g, r, equal_nan=True), (what, "layer", i // 2, "KV"[i % 2],
                                                      np.argwhere(g != r)[:4].tolist())
    assert np.array_equal(gl, rl, equal_nan=True), (what, np.argwhere(gl != rl)[:4].tolist())


def _check(m, batch, n, seed=3):
    prompts = np.random.default_rng(seed).integers(0, m.cfg.vocab, (batch, n))
    m.reset(batch)
    _stepwise(m, prompts)
    ref, token = _state(m, batch, n), m.next_tokens()
    m.reset(batch)
    out = m.generate(prompts, 1)
    _same(_state(m, batch, n), ref, (batch, n))
    assert np.array_equal(out[:, 0], token)
    print(f"batch {batch}, {n} tokens: ok", flush=True)


# Per model: token counts at the edges of the 32-token GEMM tiles, the 16-token
# q / k / v blocks, the attention's token blocks and its splits.
#  - the Qwen3 shape (splits of 144 positions), up to 17 of them;
#  - 32 splits of 16 positions, so that merge groups hold two splits each;
#  - splits of 512 positions: four 128-position halves, the softmax sums' lanes
#    taken a second time;
#  - GPT-2 on its layers kernel (batch 1, splits of 256) and on the per-op
#    kernels (other batches; one split and three); the per-op kernels of Qwen3, one
#    split and three
CASES = [
    ("qwen3-wide", QWEN_WIDE, "1", [(1, 5), (1, 145), (1, 290), (2, 161), (4, 67), (16, 21)]),
    ("qwen3-wide-long", QWEN_WIDE, "1", [(1, 2450)]),
    ("qwen3-splits-of-16", QWEN_SMALL.with_(max_positions=512), "1", [(1, 6), (1, 33), (3, 258), (1, 500)]),
    ("qwen3-splits-of-512", QWEN_SMALL.with_(max_positions=16384), "1", [(1, 130), (1, 257), (2, 700)]),
    ("gpt2-wide", GPT2_WIDE, "1", [(1, 5), (1, 129), (1, 257), (1, 700), (2, 66), (16, 33)]),
    ("gpt2-small", GPT2_SMALL_TEST, "1", [(1, 7), (1, 100), (3, 65)]),
    ("gpt2-d128", GPT2_SMALL_TEST.with_(heads=2, kv_heads=2, head_dim=128), "1", [(1, 90), (3, 65)]),
    ("gpt2-odd-quarters", GPT2_SMALL_TEST.with_(hidden=384, heads=6, kv_heads=6, intermediate=640), "1",
     [(1, 90), (3, 65)]),
    ("qwen3-per-op", QWEN_SMALL, "0", [(1, 7), (1, 130), (3, 65)]),
    ("qwen3-per-op-mha", QWEN_SMALL.with_(heads=2, hidden=512), "1", [(2, 66)]),
    ("qwen3-per-op-splits", QWEN_SMALL.with_(max_positions=2100), "0", [(2, 720)]),
    ("gpt2-per-op-splits", GPT2_SMALL_TEST.with_(max_positions=2100), "1", [(1, 1060), (2, 66)]),
]


@pytest.mark.parametrize("name,cfg,layers_kernel,sizes", CASES, ids=[c[0] for c in CASES])
def test_prompt_pass_is_the_steps(ctx, monkeypatch, name, cfg, layers_kernel, sizes):
    monkeypatch.setenv("STRICT_HIP_LLM_LAYERS", layers_kernel)
    with _model(ctx, cfg) as m:
        for batch, n in sizes:
            _check(m, batch, n)


@pytest.mark.parametrize("cfg", [QWEN_SMALL, GPT2_SMALL_TEST], ids=["qwen3", "gpt2"])
@pytest.mark.parametrize("batch", [1, 2])
def test_prompt_pass_after_cached_tokens_is_the_steps(ctx, cfg, batch):
    # (V^T stores that start at positions which are no multiple of 8)
    rng = np.random.default_rng(5)
    with _model(ctx, cfg) as m:
        for first, n in ((1, 20), (5, 64), (90, 75)):
            head, mid, tail = (rng.integers(0, cfg.vocab, (batch, k)) for k in (first, n, 33))
            m.reset(batch)
            _stepwise(m, np.concatenate([head, mid, tail], axis=1))
            ref = _state(m, batch, first + n + 33)
            m.reset(batch)
            _stepwise(m, head)
            m.generate(mid, 1)
            m.generate(tail, 1)
            _same(_state(m, batch, first + n + 33), ref, (first, n))


@pytest.mark.parametrize("cfg", [QWEN_WIDE, GPT2_WIDE], ids=["qwen3", "gpt2"])
def test_prompt_in_chunks_is_the_steps(ctx, cfg):
    # 16 x 300 rows: more than a pass takes at once, so chunks of 256 positions
    with _model(ctx, cfg) as m:
        _check(m, 16, 300)


@pytest.mark.parametrize("cfg", [QWEN_SMALL, GPT2_SMALL_TEST], ids=["qwen3", "gpt2"])
@pytest.mark.parametrize("batch", [1, 2])
def test_a_value_that_overflows_fp16_stays_with_its_token(ctx, cfg, batch):
    # one token's V is infinite (its value rows see an embedding that no other
    # token has): the tokens before it must not see that, as they do not in steps
    with _model(ctx, cfg) as m:
        d, heads, kvh = cfg.head_dim, cfg.heads, cfg.kv_heads
        rng = np.random.default_rng(1)
        head = rng.normal(0, 0.02, (cfg.vocab_pad, cfg.hidden)).astype(np.float32)
        head[:, 0] = 0.0
        head[7] = 0.0
        head[7, 0] = 1.0  # token 7 alone points along axis 0
        m.load_linear("head", 0, head)
        qkv = rng.normal(0, 0.02, (cfg.qkv_rows, cfg.hidden)).astype(np.float32)
        qkv[(heads + kvh) * d:, 0] = 3e4
        m.load_linear("qkv", 0, qkv)
        prompts = rng.integers(8, cfg.vocab, (batch, 60))
        prompts[:, 37] = 7
        m.reset(batch)
        _stepwise(m, prompts)
        ref = _state(m, batch, 60)
        assert not np.isfinite(ref[0][1][0, :, 37]).all(), "the case does not overflow"
        assert np.isfinite(ref[0][2][0, :, :37]).all()
        m.reset(batch)
        m.generate(prompts, 1)
        _same(_state(m, batch, 60), ref, "overflow")
