"""sh_llm_generate's one-pass prompt against the same prompt token by token
(sh_llm_step, itself checked against the oracle in test_gpu_llm.py): KV
caches of every layer, logits, lengths and history.

The pass sums in the steps' own order and leaves their bits
(test_gpu_prompt_exact.py). The bounds here are those of any order of sums: a
K or V value is one fp16 rounding (2^-11) of a value whose inputs were rounded
to fp16 twice per layer, and another order flips some of those roundings by one
step (2^-10). 4 x 2^-10 in the 2-norm and the attention bar of test_gpu_llm.py
(1e-2 of the largest value) for the maximum hold; a wrong position, head or
mask is off by order 1."""
import numpy as np
import pytest

import strict_amd
from strict_amd import llm
from test_gpu_llm import GPT2_SMALL_TEST, LOGIT_REL_TOL, QWEN_SMALL, _randomize_small_params

pytestmark = pytest.mark.gpu


def _caches(m, batch, n):
    """K and V [layer][batch, kv head, position < n, dim] as fp32."""
    c = m.cfg
    vt = (c.max_positions + 15) // 16 * 16
    transposed = c.arch == llm.QWEN3 and m.uses_layers_kernel
    out = []
    for li in range(c.layers):
        size = c.max_batch * c.kv_heads * c.head_dim
        k = m.read("kcache", li, np.float16)[: size * c.max_positions]
        k = k.reshape(c.max_batch, c.kv_heads, c.max_positions, c.head_dim)
        if transposed:
            v = m.read("vcache", li, np.float16)[: size * vt].reshape(
                c.max_batch, c.kv_heads, c.head_dim, vt).transpose(0, 1, 3, 2)
        else:
            v = m.read("vcache", li, np.float16)[: size * c.max_positions].reshape(k.shape)
        out += [k[:batch, :, :n].astype(np.float32), v[:batch, :, :n].astype(np.float32)]
    return out


def _state(m, batch, n):
    return (_caches(m, batch, n), m.logits().copy(), m.read("lens", 0, np.int32)[:batch].copy(),
            m.read("hist", 0, np.int32).reshape(m.cfg.max_batch, -1)[:batch, :n].copy())


def _stepwise(m, prompts):
    for i in range(prompts.shape[1]):
        m.step(prompts[:, i], logits=(i == prompts.shape[1] - 1))


def _close(got, ref):
    (gc, gl, glen, gh), (rc, rl, rlen, rh) = got, ref
    assert np.array_equal(glen, rlen) and np.array_equal(gh, rh)
    for i, (g, r) in enumerate(zip(gc, rc)):
        assert np.linalg.norm(g - r) <= 4 * 2.0 ** -10 * np.linalg.norm(r), i
        assert np.max(np.abs(g - r)) <= 1e-2 * np.max(np.abs(r)), i
    assert np.max(np.abs(gl - rl)) <= LOGIT_REL_TOL * np.max(np.abs(rl))


# 7: less than a block; 17, 65, 66: edges of the 16-token q / k / v blocks and of
# the 32-token GEMM tiles; 130, 301: a partial last tile, several splits
@pytest.mark.parametrize("cfg,layers_kernel", [(QWEN_SMALL, "1"), (QWEN_SMALL, "0"),
                                               (QWEN_SMALL.with_(heads=2, hidden=512), "1"),
                                               (GPT2_SMALL_TEST, "1"),
                                               (GPT2_SMALL_TEST.with_(heads=2, kv_heads=2, head_dim=128), "1")],
                         ids=["qwen3", "qwen3-per-op", "qwen3-mha", "gpt2", "gpt2-d128"])
def test_prompt_pass_vs_steps(ctx, monkeypatch, cfg, layers_kernel):
    monkeypatch.setenv("STRICT_HIP_LLM_LAYERS", layers_kernel)
    rng = np.random.default_rng(17)
    with llm.Model(ctx, cfg.with_(max_positions=488)) as m:
        m.init_random(seed=7, stddev=0.02)
        _randomize_small_params(m, 1)
        for batch, n in ((1, 7), (3, 17), (1, 65), (2, 66), (1, 130), (4, 301)):
            prompts = rng.integers(0, cfg.vocab, (batch, n))
            m.reset(batch)
            _stepwise(m, prompts)
            ref = _state(m, batch, n)
            m.reset(batch)
            m.generate(prompts, 1)
            _close(_state(m, batch, n), ref)
            print(f"batch {batch}, {n} tokens: ok", flush=True)


@pytest.mark.parametrize("cfg", [QWEN_SMALL, GPT2_SMALL_TEST], ids=["qwen3", "gpt2"])
def test_prompt_pass_after_cached_tokens(ctx, cfg):
    # the prompt continues sequences that hold 1 .. 90 tokens already (its
    # V^T stores start at positions that are no multiple of 8), and a second
    # prompt continues the first
    rng = np.random.default_rng(5)
    with llm.Model(ctx, cfg) as m:
        m.init_random(seed=7, stddev=0.02)
        _randomize_small_params(m, 1)
        for first, n in ((1, 20), (5, 64), (90, 75)):
            head, mid, tail = (rng.integers(0, cfg.vocab, (2, k)) for k in (first, n, 33))
            m.reset(2)
            _stepwise(m, np.concatenate([head, mid, tail], axis=1))
            total = first + n + 33
            ref = _state(m, 2, total)
            m.reset(2)
            _stepwise(m, head)
            m.generate(mid, 1)
            m.generate(tail, 1)
            _close(_state(m, 2, total), ref)


# two tokens past 16-token blocks, an odd and an even number of 32-token blocks,
# one and two positions past a 128-position part and past two
@pytest.mark.parametrize("cfg", [QWEN_SMALL, GPT2_SMALL_TEST], ids=["qwen3", "gpt2"])
@pytest.mark.parametrize("batch,n", [(2, 34), (1, 97), (1, 130), (2, 162), (1, 258)])
def test_prompt_attention_block_edges(ctx, cfg, batch, n):
    prompts = np.random.default_rng(n).integers(0, cfg.vocab, (batch, n))
    with llm.Model(ctx, cfg.with_(max_positions=300)) as m:
        m.init_random(seed=7, stddev=0.02)
        _randomize_small_params(m, 1)
        m.reset(batch)
        _stepwise(m, prompts)
        ref = _state(m, batch, n)
        m.reset(batch)
        m.generate(prompts, 1)
        _close(_state(m, batch, n), ref)


def test_prompt_pass_rows_do_not_depend_on_the_batch(ctx):
    # 16 sequences of 300 tokens take the pass in chunks of 256 positions; a
    # sequence alone takes it in one: caches and logits bit for bit the same
    cfg = QWEN_SMALL.with_(max_batch=16)
    prompts = np.random.default_rng(8).integers(0, cfg.vocab, (16, 300))
    with llm.Model(ctx, cfg) as m:
        m.init_random(seed=7, stddev=0.02)
        _randomize_small_params(m, 1)
        m.reset(16)
        m.generate(prompts, 1)
        caches, logits, _, hist = _state(m, 16, 300)
        assert np.array_equal(hist, prompts)
        for b in (0, 9, 15):
            m.reset(1)
            m.generate(prompts[b:b + 1], 1)
            one, l1, _, _ = _state(m, 1, 300)
            for x, y in zip(one, caches):
                assert np.array_equal(x[0], y[b]), b
            assert np.array_equal(l1[0], logits[b]), b


def test_prompt_with_a_token_outside_the_vocabulary_is_refused(ctx):
    cfg = QWEN_SMALL
    prompt = np.random.default_rng(2).integers(0, cfg.vocab, (1, 24))
    prompt[0, 13] = cfg.vocab
    with llm.Model(ctx, cfg) as m:
        m.init_random(seed=7, stddev=0.02)
        m.reset(1)
        with pytest.raises(strict_amd.StrictHipError) as e:
            m.generate(prompt, 2)
        assert "outside the vocabulary" in str(e.value)
        ctx.sync()
        assert m.read("lens", 0, np.int32)[0] == 13  # the tokens before it went through
