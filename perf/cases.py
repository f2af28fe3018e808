"""The framework's work as its users call it: sizes, inputs, one pass, and what
that pass computes in 64 bits.

A case is a dict of plain values with a "kind":

  elementwise  sigmoid / binary / saxpy of n fp32 values
  image        brightness and 5x5 box blur of an 8-bit image, separate or fused
  gemm_bf16    C = A B, bf16
  gemm_fp8     C = sa sb^T (A Bt^T), OCP E4M3 bytes with row / column scales
  attention    one layer's grouped-query decode attention over fp16 caches
  block        the fp32 pieces between a decoder block's linears: norm, RoPE, SwiGLU / GELU
  head         LM head (FP8 weights, fp16 activations) and greedy argmax
  llm          a whole model: a prompt through `generate`, then `steps` known
               tokens through `step` (scoring a continuation), logits out

Buffers are torch tensors registered with the library context; every pass runs
on the context's stream and nothing here waits for it.
"""
import math

import numpy as np
import torch

import strict_amd
from strict_amd import llm

_CONTEXT = None


def _context():
    global _CONTEXT
    if _CONTEXT is None:
        _CONTEXT = strict_amd.Context(0)
    return _CONTEXT


class _State:
    """What a program holds before the call: registered buffers, perhaps a
    model, the call itself and the outputs it fills."""

    def __init__(self):
        self.ctx = _context()
        self.registered = []
        self.owner = None
        self.call = None
        self.outputs = None

    def buf(self, t):
        """The device address of a contiguous tensor the context may use."""
        assert t.is_contiguous() and t.is_cuda
        self.ctx.register_external(t.data_ptr(), t.numel() * t.element_size())
        self.registered.append(t)
        return t.data_ptr()

    def __del__(self):
        try:
            self.ctx.sync()
            for t in self.registered:
                self.ctx.unregister_external(t.data_ptr())
        except Exception:
            pass


class _Owner:
    """Frees a model's device memory when the last state or output of it goes."""

    def __init__(self, model):
        self.model = model

    def __del__(self):
        try:
            self.model.close()  # waits for the context's stream
        except Exception:
            pass


class _DeviceArray:
    """Device memory of a model as something torch can wrap; the tensor made
    of it keeps this object, and with it the model."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape),
                                         "typestr": typestr, "version": 2}

    def tensor(self):
        t = torch.as_tensor(self, device="cuda")
        assert t.data_ptr() == self.__cuda_array_interface__["data"][0]
        return t


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, std=1.0, mean=0.0):
    return torch.randn(*shape, generator=g, device="cuda") * std + mean


# ---- the cases ----------------------------------------------------------------

def listed():
    return [
        # the smallest call: the 10,000-value sigmoid; launch and host latency
        {"name": "sigmoid_10k", "kind": "elementwise", "op": "sigmoid", "n": 10_000},
        # the sigmoid workload of the benchmark, 2^24 values; a plain HBM stream
        {"name": "sigmoid_16m", "kind": "elementwise", "op": "sigmoid", "n": 1 << 24},
        # the image workload of the benchmark in its fused form: brighten, then blur
        {"name": "brightness_blur_rgba_4096", "kind": "image", "op": "fused", "width": 4096,
         "height": 4096, "channels": 4, "delta": 40, "all_channels": False, "mode": 0},
        # an RGB photograph of an odd size, the reference's own blur rule
        {"name": "blur_rgb_1919x1079", "kind": "image", "op": "blur", "width": 1919,
         "height": 1079, "channels": 3, "delta": 0, "all_channels": False, "mode": 1},
        # the GEMM workload of the benchmark
        {"name": "gemm_bf16_4096", "kind": "gemm_bf16", "m": 4096, "n": 4096, "k": 4096},
        # a GEMM whose sizes are nobody's tile
        {"name": "gemm_bf16_1000x1003x517", "kind": "gemm_bf16", "m": 1000, "n": 1003, "k": 517},
        # 517 tokens through the gate/up linear of the Qwen3 shape, quantized both sides
        {"name": "gemm_fp8_517x6144x1024", "kind": "gemm_fp8", "m": 517, "n": 6144, "k": 1024},
        # decode attention of one layer of the Qwen3 shape, 4 sequences of different lengths
        {"name": "attn_decode_b4_kv4096", "kind": "attention", "batch": 4, "heads": 16,
         "kv_heads": 8, "head_dim": 128, "max_positions": 4352, "longest": 4096},
        # the pieces between the linears of one Qwen3-shaped block, 512 tokens
        {"name": "block_qwen3_512", "kind": "block", "arch": "qwen3", "rows": 512, "hidden": 1024,
         "heads": 16, "head_dim": 128, "intermediate": 3072},
        # LM head of the Qwen3 shape and the greedy token of 16 sequences
        {"name": "head_greedy_b16", "kind": "head", "batch": 16, "k": 1024, "n": 151936},
        # the Qwen3 shape: a 1,024-token prompt, then 32 tokens of decode
        {"name": "qwen3_prompt1024_decode32", "kind": "llm", "arch": "qwen3", "layers": 28,
         "batch": 1, "prompt": 1024, "steps": 32},
        # GPT-2 small: the benchmark's 128-token prompt, then 64 tokens of decode
        {"name": "gpt2_prompt128_decode64", "kind": "llm", "arch": "gpt2", "layers": 12,
         "batch": 1, "prompt": 128, "steps": 64},
    ]


def _log_int(rng, lo, hi):
    """A whole number spread evenly over the logarithm of lo .. hi."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["elementwise", "image", "image", "gemm_bf16", "gemm_bf16", "gemm_fp8",
                       "gemm_fp8", "attention", "block", "head", "llm", "llm"])
    if kind == "elementwise":
        return {"kind": kind, "op": rng.choice(["sigmoid", "add", "multiply", "saxpy"]),
                "n": _log_int(rng, 1_000, 1 << 24)}
    if kind == "image":
        width = _log_int(rng, 64, 4096)
        return {"kind": kind, "op": rng.choice(["brightness", "blur", "fused"]), "width": width,
                "height": _log_int(rng, 48, 4096), "channels": rng.choice([1, 3, 3, 4, 4]),
                "delta": rng.choice([-40, 40, 17, 0]), "all_channels": rng.random() < 0.25,
                "mode": rng.choice([0, 1])}
    if kind in ("gemm_bf16", "gemm_fp8"):
        # a third of the sizes on multiples of 64, as weights have; the rest as they come
        sizes = [_log_int(rng, 16, 4096) for _ in range(3)]
        sizes = [max(64, s // 64 * 64) if rng.random() < 0.34 else s for s in sizes]
        return {"kind": kind, "m": sizes[0], "n": sizes[1], "k": sizes[2]}
    if kind == "attention":
        head_dim = rng.choice([64, 128])
        heads, kv_heads = rng.choice([(16, 8), (12, 12), (32, 4), (16, 1)])
        max_positions = _log_int(rng, 128, 8192)
        return {"kind": kind, "batch": rng.choice([1, 2, 4, 8, 16]), "heads": heads,
                "kv_heads": kv_heads, "head_dim": head_dim, "max_positions": max_positions,
                "longest": rng.randint(max_positions // 2, max_positions)}
    if kind == "block":
        arch = rng.choice(["qwen3", "gpt2"])
        return {"kind": kind, "arch": arch, "rows": _log_int(rng, 1, 2048),
                "hidden": 1024 if arch == "qwen3" else 768, "heads": 16 if arch == "qwen3" else 12,
                "head_dim": 128 if arch == "qwen3" else 64, "intermediate": 3072}
    if kind == "head":
        return {"kind": kind, "batch": rng.randint(1, 16), "k": rng.choice([768, 1024, 2048]),
                "n": _log_int(rng, 2_000, 151_936) // 16 * 16}
    arch = rng.choice(["qwen3", "gpt2"])
    batch = rng.choice([1, 1, 2, 4])
    return {"kind": kind, "arch": arch,
            "layers": rng.randint(2, 12 if arch == "gpt2" else 28), "batch": batch,
            "prompt": _log_int(rng, 8, 640 // batch), "steps": rng.randint(0, 24)}


# ---- inputs ---------------------------------------------------------------------

def _quantize_rows(w):
    """Per-row OCP E4M3 bytes and fp32 scales of w, as a weight file holds them."""
    scale = w.abs().amax(dim=1).clamp_min(1e-30) / 448.0
    return (w / scale[:, None]).to(torch.float8_e4m3fn), scale


def _inputs(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "elementwise":
        n = case["n"]
        x = torch.rand(n, generator=g, device="cuda") * 16 - 8
        if case["op"] == "sigmoid":
            return {"x": x}
        return {"x": x, "y": _randn(g, n, std=3.0)}
    if kind == "image":
        size = case["width"] * case["height"] * case["channels"]
        return {"x": torch.randint(0, 256, (size,), generator=g, device="cuda", dtype=torch.uint8)}
    if kind == "gemm_bf16":
        m, n, k = case["m"], case["n"], case["k"]
        return {"a": _randn(g, m, k, std=0.02).bfloat16(), "b": _randn(g, k, n, std=0.02).bfloat16()}
    if kind == "gemm_fp8":
        m, n, k = case["m"], case["n"], case["k"]
        a, sa = _quantize_rows(_randn(g, m, k))
        b, sb = _quantize_rows(_randn(g, n, k, std=0.02))
        return {"a": a, "sa": sa, "b": b, "sb": sb}
    if kind == "attention":
        b, h, kvh, d, p = (case[x] for x in ("batch", "heads", "kv_heads", "head_dim", "max_positions"))
        lengths = torch.randint(max(1, case["longest"] // 3), case["longest"] + 1, (b,), generator=g,
                                device="cuda", dtype=torch.int32)
        lengths[0] = case["longest"]
        return {"q": _randn(g, b, h, d), "k": _randn(g, b, kvh, p, d).half(),
                "v": _randn(g, b, kvh, p, d).half(), "lengths": lengths}
    if kind == "block":
        r, hid, h, d, i = (case[x] for x in ("rows", "hidden", "heads", "head_dim", "intermediate"))
        return {"x": _randn(g, r, hid, std=1.5, mean=0.1), "gain": _randn(g, hid, std=0.1, mean=1.0),
                "bias": _randn(g, hid, std=0.05), "q": _randn(g, r, h, d),
                "positions": torch.arange(r, device="cuda", dtype=torch.int32) + int(seed) % 1000,
                "gate": _randn(g, r, i, std=2.0), "up": _randn(g, r, i)}
    if kind == "head":
        w, s = _quantize_rows(_randn(g, case["n"], case["k"], std=0.02))
        return {"x": _randn(g, case["batch"], case["k"]).half(), "w": w, "s": s}
    raise ValueError(kind)


def _model_config(case):
    base = llm.QWEN3_0_6B if case["arch"] == "qwen3" else llm.GPT2_SMALL
    return base.with_(layers=case["layers"], max_batch=case["batch"])


def _linear_names(cfg):
    return ("qkv", "o", "gate_up", "down") if cfg.arch == llm.QWEN3 else ("qkv", "o", "fc", "proj")


def _model_weights(cfg, seed):
    """(name, layer, fp32 tensor) of every linear, then norms, biases and
    tokens' tables: what a checkpoint of the architecture holds. The FP8
    model's matrices are E4M3 values times a scale per row, so that loading
    them quantizes them to themselves."""
    g = _generator(seed)
    shapes = llm.linear_shapes(cfg)

    def matrix(name):
        rows, cols = shapes[name]
        w = _randn(g, rows, cols, std=0.02)
        if name == "head":
            w[cfg.vocab:] = 0
        if cfg.arch == llm.QWEN3:
            q, s = _quantize_rows(w)
            return q.float() * s[:, None]
        return w.half().float()

    for layer in range(cfg.layers):
        for name in _linear_names(cfg):
            yield name, layer, matrix(name)
        for name in ("norm1.g", "norm2.g"):
            yield name, layer, _randn(g, cfg.hidden, std=0.1, mean=1.0)
        if cfg.arch == llm.QWEN3:
            for name in ("q_norm", "k_norm"):
                yield name, layer, _randn(g, cfg.head_dim, std=0.1, mean=1.0)
        else:
            for name in ("norm1.b", "norm2.b"):
                yield name, layer, _randn(g, cfg.hidden, std=0.05)
            for name in _linear_names(cfg):
                yield name + ".bias", layer, _randn(g, shapes[name][0], std=0.02)
    yield "head", 0, matrix("head")
    yield "final.g", 0, _randn(g, cfg.hidden, std=0.1, mean=1.0)
    if cfg.arch == llm.GPT2:
        yield "final.b", 0, _randn(g, cfg.hidden, std=0.05)
        yield "wpe", 0, _randn(g, cfg.max_positions, cfg.hidden, std=0.02).half()


def _tokens(case, cfg, seed):
    rng = np.random.default_rng(int(seed))
    return (rng.integers(0, cfg.vocab, (case["batch"], case["prompt"]), dtype=np.int32),
            rng.integers(0, cfg.vocab, (case["steps"], case["batch"]), dtype=np.int32))


# ---- one pass ---------------------------------------------------------------------

def prepare(case, seed):
    st = _State()
    ctx, kind = st.ctx, case["kind"]
    if kind == "llm":
        _prepare_model(st, case, seed)
        return st
    t = _inputs(case, seed)
    p = {name: st.buf(x) for name, x in t.items()}

    def out(shape, dtype):
        x = torch.zeros(shape, dtype=dtype, device="cuda")
        return x, st.buf(x)

    if kind == "elementwise":
        n = case["n"]
        y, py = out(n, torch.float32)
        if case["op"] == "sigmoid":
            st.call = lambda: ctx.sigmoid(p["x"], py, n)
        elif case["op"] == "saxpy":
            st.call = lambda: ctx.saxpy(1.7, p["x"], p["y"], py, n)
        else:
            op = strict_amd.ADD if case["op"] == "add" else strict_amd.MULTIPLY
            st.call = lambda: ctx.binary(op, p["x"], p["y"], py, n)
        st.outputs = y
    elif kind == "image":
        w, h, c = case["width"], case["height"], case["channels"]
        flags = strict_amd.BRIGHTNESS_ALL_CHANNELS if case["all_channels"] else 0
        y, py = out(w * h * c, torch.uint8)
        if case["op"] == "brightness":
            st.call = lambda: ctx.adjust_brightness(p["x"], py, w, h, c, case["delta"], flags)
        elif case["op"] == "blur":
            st.call = lambda: ctx.box_blur5(p["x"], py, w, h, c, case["mode"])
        else:
            st.call = lambda: ctx.brightness_blur5(p["x"], py, w, h, c, case["delta"], flags,
                                                   case["mode"])
        st.outputs = y
    elif kind == "gemm_bf16":
        m, n, k = case["m"], case["n"], case["k"]
        y, py = out((m, n), torch.bfloat16)
        st.call = lambda: ctx.gemm_bf16(p["a"], p["b"], py, m, n, k)
        st.outputs = y
    elif kind == "gemm_fp8":
        m, n, k = case["m"], case["n"], case["k"]
        y, py = out((m, n), torch.bfloat16)
        st.call = lambda: ctx.gemm_fp8(p["a"], p["sa"], p["b"], p["sb"], py, m, n, k)
        st.outputs = y
    elif kind == "attention":
        b, h, kvh, d, mp = (case[x] for x in ("batch", "heads", "kv_heads", "head_dim", "max_positions"))
        y, py = out((b, h, d), torch.float32)
        st.call = lambda: ctx.attn_decode(p["q"], p["k"], p["v"], p["lengths"], py, b, h, kvh, d, mp,
                                          1.0 / math.sqrt(d))
        st.outputs = y
    elif kind == "block":
        _prepare_block(st, case, t, p, out)
    else:
        b, k, n = case["batch"], case["k"], case["n"]
        tiled, pt = out((n, k), torch.uint8)
        torch.cuda.synchronize()  # the context's stream packs what torch's has made
        ctx.pack_e4m3_tiles(p["w"], pt, n, k)
        y, py = out((b, n), torch.float32)
        i, pi = out(b, torch.int32)

        def call():
            ctx.gemv_w8a16(p["x"], pt, p["s"], py, b, k, n)
            ctx.argmax(py, b, n, pi)
        st.call = call
        st.outputs = {"logits": y, "token": i}
    return st


def _prepare_block(st, case, t, p, out):
    """Norm, RoPE of the queries and the MLP's activation; the query rows are
    rotated from a copy, as RoPE works in place and a pass starts from q."""
    ctx = st.ctx
    r, hid, h, d, i = (case[x] for x in ("rows", "hidden", "heads", "head_dim", "intermediate"))
    y, py = out((r, hid), torch.float32)
    act, pact = out((r, i), torch.float32)
    if case["arch"] == "gpt2":
        def call():
            ctx.layernorm(p["x"], p["gain"], p["bias"], py, r, hid, 1e-5)
            ctx.gelu(p["gate"], pact, r * i)
        st.call = call
        st.outputs = {"norm": y, "act": act}
        return
    q, pq = out((r, h, d), torch.float32)
    src = strict_amd.DeviceVariable(ctx, p["q"], r * h * d * 4, np.float32)
    dst = strict_amd.DeviceVariable(ctx, pq, r * h * d * 4, np.float32)

    def call():
        ctx.rmsnorm(p["x"], p["gain"], py, r, hid, 1e-6)
        ctx.copy(dst, src)
        ctx.rope(pq, p["positions"], r, h, d, 1e6)
        ctx.swiglu(p["gate"], p["up"], pact, r * i)
    st.call = call
    st.outputs = {"norm": y, "q": q, "act": act}


def _prepare_model(st, case, seed):
    cfg = _model_config(case)
    m = llm.Model(st.ctx, cfg)
    owner = st.owner = _Owner(m)
    linears = set(llm.linear_shapes(cfg))
    for name, layer, w in _model_weights(cfg, seed):
        if name in linears:
            m.load_linear(name, layer, w.cpu().numpy())
        else:
            m.write(name, layer, w.cpu().numpy())
    prompt, known = _tokens(case, cfg, seed)
    b = case["batch"]

    def wrap(name, layer, shape, typestr):
        ptr, nbytes = m.tensor(name, layer)
        assert math.prod(shape) * int(typestr[2:]) <= nbytes
        return _DeviceArray(owner, ptr, shape, typestr).tensor()

    # the logits of the last token and the keys the last layer has cached
    st.outputs = {"logits": wrap("logits", 0, (b, cfg.vocab_pad), "<f4")[:, : cfg.vocab],
                  "keys": wrap("kcache", cfg.layers - 1,
                               (b, cfg.kv_heads, cfg.max_positions, cfg.head_dim), "<f2")}
    for t in st.outputs.values():
        t.owner = owner  # an output that outlives its state keeps the model

    def call():
        m.reset(b)
        m.generate(prompt, 1)
        for tokens in known:
            m.step(tokens, logits=True)
    st.call = call


def run(state):
    state.call()
    return state.outputs


# ---- what a pass cannot do without ---------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "elementwise":
        n = case["n"]
        return {"bytes": n * (8 if case["op"] == "sigmoid" else 12), "flops": 0}
    if kind == "image":
        return {"bytes": 2 * case["width"] * case["height"] * case["channels"], "flops": 0}
    if kind in ("gemm_bf16", "gemm_fp8"):
        m, n, k = case["m"], case["n"], case["k"]
        e = 2 if kind == "gemm_bf16" else 1
        return {"bytes": e * (m * k + k * n) + 2 * m * n, "flops": 2 * m * n * k}
    if kind == "attention":
        b, h, kvh, d = (case[x] for x in ("batch", "heads", "kv_heads", "head_dim"))
        # the first sequence is the longest, the others a third of it and up
        positions = case["longest"] * (1 + (b - 1) * 2 / 3)
        return {"bytes": positions * kvh * d * 4 + b * h * d * 8, "flops": positions * h * d * 4}
    if kind == "block":
        r, hid, h, d, i = (case[x] for x in ("rows", "hidden", "heads", "head_dim", "intermediate"))
        if case["arch"] == "gpt2":
            return {"bytes": 8 * r * (hid + i), "flops": 0}
        return {"bytes": r * (8 * hid + 8 * h * d + 12 * i), "flops": 0}
    if kind == "head":
        b, k, n = case["batch"], case["k"], case["n"]
        return {"bytes": n * k + 4 * n + 2 * b * k + 4 * b * n, "flops": 2 * b * n * k}
    cfg = _model_config(case)
    b, prompt, steps = case["batch"], case["prompt"], case["steps"]
    shapes = llm.linear_shapes(cfg)
    params = cfg.layers * sum(r * c for name, (r, c) in shapes.items() if name != "head")
    head = cfg.vocab * cfg.hidden
    one = llm.decode_step_bytes(cfg, b, prompt + steps / 2.0)
    kv_token = cfg.layers * 2 * cfg.kv_heads * cfg.head_dim
    pairs = b * prompt * prompt / 2 + steps * b * (prompt + steps / 2.0)
    return {
        # every weight once for the prompt and once for a decode step, the caches
        # written by the prompt and read by the steps
        "bytes": one["weights"] + b * prompt * kv_token * 2 + steps * one["total"],
        "flops": 2 * params * b * (prompt + steps) + 2 * head * b * (1 + steps)
        + pairs * cfg.layers * cfg.heads * cfg.head_dim * 4,
    }


def tolerance(case):
    """About four times what a correct path is off the 64-bit result, or two
    correct ones off each other, whichever is the larger (measured)."""
    kind = case["kind"]
    if kind == "image":
        return "exact"
    if kind == "elementwise":
        # fp32 exp, one add and one divide, each rounded once; the others one
        # rounding: 4e-8 off the exact result
        return {"rel": 2e-7, "max": 1e-6}
    if kind in ("gemm_bf16", "gemm_fp8"):
        # rounding to bf16 alone is 1.7e-3 off the exact result; a sum in
        # another order moves a few values by one bf16 step (2^-8)
        return {"rel": 4e-3, "max": 2e-2}
    if kind == "attention":
        # fp32 scores, exponentials and sums: 4e-7 off
        return {"rel": 2e-6, "max": 2e-5}
    if kind == "block":
        # one rounding per fp32 operation: 5e-8 off
        return {"rel": 3e-7, "max": 1e-5}
    if kind == "head":
        # fp32 sums of exact products: 1e-7 off
        return {"rel": 6e-7, "max": 1e-5}
    # fp16 activations, rounded again in every layer: 9e-4 off, and two correct
    # orders of the sums differ as much
    return {"rel": 4e-3, "max": 4e-2}


# ---- the same in 64 bits ---------------------------------------------------------------

def exact(case, seed):
    kind = case["kind"]
    if kind == "llm":
        return _exact_model(case, seed)
    t = _inputs(case, seed)
    if kind == "elementwise":
        x = t["x"].double()
        if case["op"] == "sigmoid":
            return torch.sigmoid(x)
        y = t["y"].double()
        if case["op"] == "saxpy":
            return float(np.float32(1.7)) * x + y
        return x + y if case["op"] == "add" else x * y
    if kind == "image":
        return _exact_image(case, t["x"])
    if kind == "gemm_bf16":
        return t["a"].double() @ t["b"].double()
    if kind == "gemm_fp8":
        y = t["a"].double() @ t["b"].double().T
        return y * t["sa"].double()[:, None] * t["sb"].double()[None, :]
    if kind == "attention":
        return _exact_attention(case, t)
    if kind == "block":
        return _exact_block(case, t)
    y = t["x"].double() @ (t["w"].double() * t["s"].double()[:, None]).T
    return {"logits": y, "token": None}


def _exact_image(case, x):
    """Whole bytes, computed in whole numbers."""
    w, h, c = case["width"], case["height"], case["channels"]
    img = x.reshape(h, w, c).to(torch.int32)
    if case["op"] != "blur":
        # the fourth byte of a pixel passes through unless asked for
        last = c if case["all_channels"] or c < 4 else 3
        img[..., :last] = (img[..., :last] + case["delta"]).clamp(0, 255)
    if case["op"] == "brightness":
        return img.to(torch.uint8).reshape(-1)

    def windows(v, axis):
        n = v.shape[axis]
        at = torch.arange(n, device=v.device)
        total = torch.zeros_like(v)
        for k in range(-2, 3):
            idx = at + k
            part = v.index_select(axis, idx.clamp(0, n - 1))
            if case["mode"] == 1:  # taps outside the image are left out
                inside = ((idx >= 0) & (idx < n)).to(v.dtype)
                shape = [1] * v.dim()
                shape[axis] = n
                part = part * inside.reshape(shape)
            total = total + part
        return total

    total = windows(windows(img, 0), 1)
    if case["mode"] == 0:
        out = (total + 12) // 25
    else:
        out = total // windows(windows(torch.ones_like(img), 0), 1)
    return out.to(torch.uint8).reshape(-1)


def _exact_attention(case, t):
    b, h, kvh, d = (case[x] for x in ("batch", "heads", "kv_heads", "head_dim"))
    out = torch.zeros(b, h, d, dtype=torch.float64, device="cuda")
    for i in range(b):
        n = int(t["lengths"][i])
        q = t["q"][i].double().reshape(kvh, h // kvh, d) / math.sqrt(d)
        s = q @ t["k"][i, :, :n].double().transpose(1, 2)
        out[i] = (torch.softmax(s, dim=-1) @ t["v"][i, :, :n].double()).reshape(h, d)
    return out


def _rotate(x, positions, theta):
    """Rotate-half RoPE of x [tokens, heads, d]; the angle is by definition an
    fp32 product of the position and the fp32 inverse frequency."""
    d = x.shape[-1]
    inv = torch.tensor([float(np.float32(theta)) ** (-2.0 * i / d) for i in range(d // 2)],
                       dtype=torch.float64, device="cuda").float()
    angle = (positions.float()[:, None] * inv[None, :]).double()[:, None, :]
    a, b = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], dim=-1)


def _rms(x, gain, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gain


def _layer(x, gain, bias, eps):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gain + bias


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _exact_block(case, t):
    x, gain = t["x"].double(), t["gain"].double()
    if case["arch"] == "gpt2":
        return {"norm": _layer(x, gain, t["bias"].double(), 1e-5), "act": _gelu(t["gate"].double())}
    return {"norm": _rms(x, gain, 1e-6), "q": _rotate(t["q"].double(), t["positions"], 1e6),
            "act": torch.nn.functional.silu(t["gate"].double()) * t["up"].double()}


def _exact_model(case, seed):
    cfg = _model_config(case)
    qwen = cfg.arch == llm.QWEN3
    h, kvh, d, b = cfg.heads, cfg.kv_heads, cfg.head_dim, case["batch"]
    layers, top = [{} for _ in range(cfg.layers)], {}
    for name, layer, w in _model_weights(cfg, seed):
        (top if name in ("head", "final.g", "final.b", "wpe") else layers[layer])[name] = w
    prompt, known = _tokens(case, cfg, seed)
    tokens = torch.from_numpy(np.concatenate([prompt, known.T], axis=1).astype(np.int64)).to("cuda")
    n = tokens.shape[1]
    positions = torch.arange(n, device="cuda")
    logits = torch.zeros(b, cfg.vocab, dtype=torch.float64, device="cuda")
    keys = torch.zeros(b, kvh, cfg.max_positions, d, dtype=torch.float64, device="cuda")
    hidden = torch.full((n, n), float("-inf"), dtype=torch.float64, device="cuda").triu(1)
    for row in range(b):
        x = top["head"][tokens[row]].double()
        if not qwen:
            x = x + top["wpe"][:n].double()
        for L in layers:
            W = {name: w.double() for name, w in L.items()}

            def linear(v, name):
                y = v @ W[name].T
                return y if qwen else y + W[name + ".bias"]

            def norm(v, name):
                if qwen:
                    return _rms(v, W[name + ".g"], cfg.norm_eps)
                return _layer(v, W[name + ".g"], W[name + ".b"], cfg.norm_eps)

            qkv = linear(norm(x, "norm1"), "qkv")
            q = qkv[:, : h * d].reshape(n, h, d)
            k = qkv[:, h * d: (h + kvh) * d].reshape(n, kvh, d)
            v = qkv[:, (h + kvh) * d:].reshape(n, kvh, d)
            if qwen:
                q = _rotate(_rms(q, W["q_norm"], cfg.norm_eps), positions, cfg.rope_theta)
                k = _rotate(_rms(k, W["k_norm"], cfg.norm_eps), positions, cfg.rope_theta)
            k, v = k.transpose(0, 1), v.transpose(0, 1)
            keys[row, :, :n] = k
            rep = h // kvh
            s = q.transpose(0, 1) @ k.repeat_interleave(rep, 0).transpose(1, 2) / math.sqrt(d) + hidden
            o = torch.softmax(s, dim=-1) @ v.repeat_interleave(rep, 0)
            x = x + linear(o.transpose(0, 1).reshape(n, h * d), "o")
            y = norm(x, "norm2")
            if qwen:
                gate, up = linear(y, "gate_up").split(cfg.intermediate, dim=1)
                x = x + linear(torch.nn.functional.silu(gate) * up, "down")
            else:
                x = x + linear(_gelu(linear(y, "fc")), "proj")
        last = x[-1:]
        if qwen:
            last = _rms(last, top["final.g"].double(), cfg.norm_eps)
        else:
            last = _layer(last, top["final.g"].double(), top["final.b"].double(), cfg.norm_eps)
        logits[row] = (last @ top["head"].double().T)[0, : cfg.vocab]
    return {"logits": logits, "keys": keys}
