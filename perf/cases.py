"""The workloads this library's speed is measured on: what a program calls through its public entry
points (autokernel_amd.kernels.get(op), and the model plug-in), over the range of sizes it calls
them with.

listed() names twelve of them; draw(rng) makes more of the same ranges. prepare(case, seed) makes
what the program holds before the call, run(state) is one call, exact(case, seed) the same result in
64-bit arithmetic by plain torch, work(case) the bytes and operations the call cannot do without
and tolerance(case) how far two correct implementations at the same precision may lie apart.

Sizes are the model shapes of this package (LlamaModel7B: 4096 wide, 32 query and 8 KV heads of 128,
FFN 11008, vocabulary 32000; GPT-2 small: 768 wide, 12 heads of 64, vocabulary 50257) and the op
table's sweep and edge sizes (spec.KERNEL_CONFIGS).
"""
from __future__ import annotations

import math
import random

import torch

from autokernel_amd import gpt2, kernels, verify

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
GPT2_WIDTH, GPT2_HEADS, GPT2_LAYERS, GPT2_VOCAB, GPT2_BLOCK = 768, 12, 12, 50257, 1024


def listed() -> list[dict]:
    return [
        # The smallest call: the norm of one decode step (a few tokens of a 4096-wide model), run
        # twice per layer; latency is all there is.
        {"name": "rmsnorm_decode", "op": "rmsnorm", "dtype": "bf16", "rows": 8, "cols": 4096},
        # A ragged activation: neither rows nor columns a multiple of anything (the op table's edge size).
        {"name": "layernorm_odd", "op": "layernorm", "dtype": "f16", "rows": 4097, "cols": 4097},
        # Probabilities over GPT-2's odd vocabulary for a batch of 4096 positions.
        {"name": "softmax_vocab", "op": "softmax", "dtype": "f16", "rows": 4096, "cols": 50257},
        # The loss of a language model's evaluation step: 4096 positions of a 32000-entry vocabulary.
        {"name": "cross_entropy_llama", "op": "cross_entropy", "dtype": "bf16", "rows": 4096, "cols": 32000},
        # Rotary embedding of a two-sequence prefill.
        {"name": "rope_prefill", "op": "rotary_embedding", "dtype": "f16", "batch": 2, "heads": 32, "seq": 2048,
         "head_dim": 128},
        # Sum over the tokens of an activation (a bias gradient, a mean over positions): a reduction
        # over a dim that is not the last.
        {"name": "reduce_tokens", "op": "reduce", "dtype": "bf16", "rows": 8192, "cols": 4096, "dim": 0},
        # One projection of a decode step: 16 sequences, one token each, against an nn.Linear weight.
        {"name": "matmul_decode", "op": "matmul", "dtype": "bf16", "m": 16, "n": 11008, "k": 4096, "layout": "nt"},
        # A full-precision product (the op table's float32 column, its primary size).
        {"name": "matmul_f32", "op": "matmul", "dtype": "f32", "m": 2048, "n": 2048, "k": 2048, "layout": "nn"},
        # The feed-forward block of a 2048-token prefill: the largest product of the 7B model.
        {"name": "mlp_prefill", "op": "fused_mlp", "dtype": "bf16", "rows": 2048, "dim": 4096, "hidden": 11008},
        # Causal grouped-query attention of a 4096-token prefill.
        {"name": "attention_prefill", "op": "flash_attention", "dtype": "f16", "batch": 1, "heads": 32, "kv_heads": 8,
         "seq_q": 4096, "seq_k": 4096, "head_dim": 128, "causal": True},
        # One decode step's attention: each of 8 sequences has one new query against its 4096 cached keys.
        {"name": "attention_decode", "op": "flash_attention", "dtype": "bf16", "batch": 8, "heads": 32, "kv_heads": 8,
         "seq_q": 1, "seq_k": 4096, "head_dim": 128, "causal": False},
        # A whole model: GPT-2 small with every op plugged in, two full contexts, logits out.
        {"name": "gpt2_forward", "op": "gpt2", "dtype": "f16", "batch": 2, "seq": 1024},
    ]


# The most one drawn case may cost: the largest listed product, fp32 product, row op and attention.
_MAX_FLOPS = {"f16": 6 * 2048 * 4096 * 11008, "bf16": 6 * 2048 * 4096 * 11008, "f32": 2 * 2048 ** 3}
_MAX_ELEMS = 4096 * 50257
_MAX_ATTN = 4 * 32 * 4096 * 4096 * 128


def _log(rng: random.Random, lo: int, hi: int) -> int:
    """An integer spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _size(rng: random.Random, lo: int, hi: int, step: int) -> int:
    """A width: mostly a multiple of `step`, as model widths are, one in four any number."""
    n = _log(rng, lo, hi)
    return n if rng.random() < 0.25 else max(lo, n // step * step)


def draw(rng: random.Random) -> dict:
    op = rng.choice(["rmsnorm", "layernorm", "softmax", "cross_entropy", "rotary_embedding", "reduce", "matmul",
                     "matmul", "fused_mlp", "flash_attention", "flash_attention", "gpt2"])
    half = rng.choice(["f16", "bf16"])
    if op in ("rmsnorm", "layernorm", "softmax", "cross_entropy", "reduce"):
        wide = 65536 if op in ("softmax", "cross_entropy") else 16384
        dtypes = ["f16", "bf16"] if op in ("rmsnorm", "reduce") else ["f16", "bf16", "f32"]
        cols = _size(rng, 128, wide, 64)
        rows = _log(rng, 1, min(32768, _MAX_ELEMS // 2 // cols))
        case = {"op": op, "dtype": rng.choice(dtypes), "rows": rows, "cols": cols}
        if op == "reduce":
            case["dim"] = rng.choice([0, 1])
        return case
    if op == "rotary_embedding":
        return {"op": op, "dtype": rng.choice(["f16", "bf16", "f32"]), "batch": _log(rng, 1, 8),
                "heads": rng.choice([4, 8, 12, 32, 40]), "seq": _log(rng, 1, 2048), "head_dim": rng.choice([64, 128])}
    if op == "matmul":
        dtype = rng.choice(["f16", "bf16", "f32"])
        while True:
            # a decode step's few tokens as often as a prefill's many
            m = _log(rng, 1, 64) if rng.random() < 0.5 else _log(rng, 64, 8192)
            n, k = _size(rng, 128, 16384, 64), _size(rng, 128, 11008, 64)
            if 2 * m * n * k <= _MAX_FLOPS[dtype]:
                return {"op": op, "dtype": dtype, "m": m, "n": n, "k": k, "layout": rng.choice(["nn", "nt"])}
    if op == "fused_mlp":
        dtype = rng.choice(["f16", "bf16", "f32"])
        while True:
            rows = _log(rng, 1, 64) if rng.random() < 0.5 else _log(rng, 64, 4096)
            dim, hidden = _log(rng, 128, 5120) // 64 * 64, _log(rng, 256, 13824) // 64 * 64
            if 6 * rows * dim * hidden <= _MAX_FLOPS[dtype]:
                return {"op": op, "dtype": dtype, "rows": rows, "dim": dim, "hidden": hidden}
    if op == "flash_attention":
        kv = rng.choice([1, 4, 8, 12, 32])
        group = rng.choice([1, 1, 4, 8]) if kv <= 8 else 1
        case = {"op": op, "dtype": half, "batch": 1, "heads": kv * group, "kv_heads": kv,
                "head_dim": rng.choice([64, 128])}
        if rng.random() < 0.5:  # decode: one query a sequence, keys and values cached
            sk = _log(rng, 16, 32768)
            most = max(1, (8 * 8 * 4096 * 128) // (kv * sk * case["head_dim"]))
            return {**case, "batch": _log(rng, 1, min(32, most)), "seq_q": 1, "seq_k": sk, "causal": False}
        s = _log(rng, 64, 4096)
        most = max(1, _MAX_ATTN // (4 * case["heads"] * s * s * case["head_dim"]))
        return {**case, "batch": _log(rng, 1, min(8, most)), "seq_q": s, "seq_k": s,
                "causal": rng.random() < 0.75}
    seq = _log(rng, 16, GPT2_BLOCK)
    return {"op": op, "dtype": half, "batch": _log(rng, 1, max(1, min(16, 2048 // seq))), "seq": seq}


# ---------------------------------------------------------------------------------- inputs
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, shape, dtype, scale: float = 1.0, mean: float = 0.0) -> torch.Tensor:
    return (torch.randn(shape, generator=g, device="cuda") * scale + mean).to(dtype)


def _gpt2_weights(g, dtype) -> dict[str, torch.Tensor]:
    """GPT-2 small's parameters: Linear and Embedding weights and biases ~ N(0, 0.02), LayerNorm
    weights 1 + N(0, 0.02)."""
    c = GPT2_WIDTH
    shapes = {"transformer.wte.weight": (GPT2_VOCAB, c), "transformer.wpe.weight": (GPT2_BLOCK, c),
              "transformer.ln_f.weight": (c,), "transformer.ln_f.bias": (c,)}
    for i in range(GPT2_LAYERS):
        for name, out, inp in (("attn.c_attn", 3 * c, c), ("attn.c_proj", c, c), ("mlp.c_fc", 4 * c, c),
                               ("mlp.c_proj", c, 4 * c)):
            shapes[f"transformer.h.{i}.{name}.weight"], shapes[f"transformer.h.{i}.{name}.bias"] = (out, inp), (out,)
        for ln in ("ln_1", "ln_2"):
            shapes[f"transformer.h.{i}.{ln}.weight"] = shapes[f"transformer.h.{i}.{ln}.bias"] = (c,)
    return {n: _randn(g, s, dtype, 0.02, 1.0 if ".ln_" in n and n.endswith("weight") else 0.0)
            for n, s in shapes.items()}


def _inputs(case: dict, seed: int) -> dict:
    """The call's tensors, from the seed alone."""
    g, dt, op = _gen(seed), DTYPES[case["dtype"]], case["op"]
    if op in ("rmsnorm", "layernorm"):
        r, c = case["rows"], case["cols"]
        w = {"x": _randn(g, (r, c), dt), "weight": _randn(g, (c,), dt, 0.02, 1.0)}
        if op == "layernorm":
            w["bias"] = _randn(g, (c,), dt, 0.02)
        return w
    if op == "softmax":
        return {"x": _randn(g, (case["rows"], case["cols"]), dt, 3.0)}
    if op == "cross_entropy":
        r, c = case["rows"], case["cols"]
        return {"logits": _randn(g, (r, c), dt, 2.0),
                "targets": torch.randint(0, c, (r,), generator=g, device="cuda")}
    if op == "rotary_embedding":
        b, h, s, d = case["batch"], case["heads"], case["seq"], case["head_dim"]
        inv = 10000.0 ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float32) / d)
        ang = torch.arange(s, device="cuda", dtype=torch.float32)[:, None] * inv
        return {"x": _randn(g, (b, h, s, d), dt), "cos": ang.cos().to(dt), "sin": ang.sin().to(dt)}
    if op == "reduce":
        return {"x": _randn(g, (case["rows"], case["cols"]), dt), "dim": case["dim"]}
    if op == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        s = 1.0 / math.sqrt(k)
        a = _randn(g, (m, k), dt)
        b = _randn(g, (n, k), dt, s).t() if case["layout"] == "nt" else _randn(g, (k, n), dt, s)
        return {"A": a, "B": b}
    if op == "fused_mlp":
        m, d, h = case["rows"], case["dim"], case["hidden"]
        return {"x": _randn(g, (m, d), dt), "w_gate": _randn(g, (h, d), dt, 0.02), "w_up": _randn(g, (h, d), dt, 0.02),
                "w_down": _randn(g, (d, h), dt, 0.02)}
    if op == "flash_attention":
        b, d = case["batch"], case["head_dim"]
        return {"Q": _randn(g, (b, case["heads"], case["seq_q"], d), dt),
                "K": _randn(g, (b, case["kv_heads"], case["seq_k"], d), dt),
                "V": _randn(g, (b, case["kv_heads"], case["seq_k"], d), dt), "causal": case["causal"]}
    return {"weights": _gpt2_weights(g, dt),
            "ids": torch.randint(0, GPT2_VOCAB, (case["batch"], case["seq"]), generator=g, device="cuda")}


def prepare(case: dict, seed: int):
    inputs = _inputs(case, seed)
    if case["op"] != "gpt2":
        return kernels.get(case["op"]), inputs
    with torch.device("cuda"):
        model = gpt2.GPT2(GPT2_VOCAB, GPT2_BLOCK, GPT2_LAYERS, GPT2_HEADS, GPT2_WIDTH).to(DTYPES[case["dtype"]])
    missing, unexpected = model.load_state_dict(inputs["weights"], strict=False)  # lm_head.weight is wte's, masks stay
    assert not unexpected and all(n == "lm_head.weight" or n.endswith("attn.bias") for n in missing), missing
    model.eval()
    verify.OptimizedModelContext(model, verify.ALL_KERNELS).__enter__()  # plugged in for the program's life

    def forward(ids):
        with torch.no_grad():
            return model(ids)
    return forward, {"ids": inputs["ids"]}


def run(state):
    fn, args = state
    return fn(**args)


# ---------------------------------------------------------------------------------- 64-bit results
def _exact_gpt2(w: dict, ids: torch.Tensor) -> torch.Tensor:
    F = torch.nn.functional
    w = {n: t.double() for n, t in w.items()}
    b, t = ids.shape
    c, h = GPT2_WIDTH, GPT2_HEADS

    def linear(x, name):
        return x @ w[name + ".weight"].t() + w[name + ".bias"]

    def norm(x, name):
        return F.layer_norm(x, (c,), w[name + ".weight"], w[name + ".bias"])

    x = w["transformer.wte.weight"][ids] + w["transformer.wpe.weight"][:t]
    future = torch.ones(t, t, dtype=torch.bool, device=ids.device).triu(1)
    for i in range(GPT2_LAYERS):
        p = f"transformer.h.{i}."
        q, k, v = (y.view(b, t, h, c // h).transpose(1, 2).contiguous()
                   for y in linear(norm(x, p + "ln_1"), p + "attn.c_attn").split(c, 2))
        s = (q @ k.transpose(2, 3).contiguous() / math.sqrt(c // h)).masked_fill(future, -math.inf)
        x = x + linear((s.softmax(-1) @ v).transpose(1, 2).reshape(b, t, c), p + "attn.c_proj")
        x = x + linear(F.gelu(linear(norm(x, p + "ln_2"), p + "mlp.c_fc")), p + "mlp.c_proj")
    return norm(x, "transformer.ln_f") @ w["transformer.wte.weight"].t()


def _exact_attention(q, k, v, causal):
    group = q.shape[1] // k.shape[1]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    future = torch.ones(q.shape[2], k.shape[2], dtype=torch.bool, device=q.device).triu(1) if causal else None
    for b in range(q.shape[0]):
        for hk in range(k.shape[1]):
            kd, vd = k[b, hk].double(), v[b, hk].double()
            for h in range(hk * group, (hk + 1) * group):
                s = q[b, h].double() @ kd.t().contiguous() * q.shape[3] ** -0.5
                if causal:
                    s = s.masked_fill(future, -math.inf)
                out[b, h] = s.softmax(-1) @ vd
    return out


def exact(case: dict, seed: int):
    i, op = _inputs(case, seed), case["op"]
    if op == "gpt2":
        return _exact_gpt2(i["weights"], i["ids"])
    if op == "flash_attention":
        return _exact_attention(i["Q"], i["K"], i["V"], i["causal"])
    d = {n: t.double() if isinstance(t, torch.Tensor) and t.is_floating_point() else t for n, t in i.items()}
    if op == "rmsnorm":
        x = d["x"]
        return x / (x.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt() * d["weight"]
    if op == "layernorm":
        return torch.nn.functional.layer_norm(d["x"], (case["cols"],), d["weight"], d["bias"], 1e-5)
    if op == "softmax":
        return d["x"].softmax(-1)
    if op == "cross_entropy":
        return torch.nn.functional.cross_entropy(d["logits"], d["targets"])
    if op == "rotary_embedding":
        a, b, c, s = d["x"][..., 0::2], d["x"][..., 1::2], d["cos"], d["sin"]
        return torch.stack((a * c - b * s, a * s + b * c), -1).flatten(-2)
    if op == "reduce":
        return d["x"].sum(d["dim"])
    if op == "matmul":
        return d["A"] @ d["B"].contiguous()
    g, u = d["x"] @ d["w_gate"].t().contiguous(), d["x"] @ d["w_up"].t().contiguous()
    return (torch.nn.functional.silu(g) * u) @ d["w_down"].t().contiguous()


# ---------------------------------------------------------------------------------- bounds
def work(case: dict) -> dict:
    op, e = case["op"], 4 if case["dtype"] == "f32" else 2
    if op in ("rmsnorm", "layernorm", "softmax", "cross_entropy", "reduce"):
        r, c = case["rows"], case["cols"]
        extra = {"rmsnorm": r * c + c, "layernorm": r * c + 2 * c, "softmax": r * c, "cross_entropy": 1,
                 "reduce": c if case.get("dim") == 0 else r}[op]
        ops = {"rmsnorm": 4, "layernorm": 7, "softmax": 4, "cross_entropy": 3, "reduce": 1}[op]
        return {"bytes": (r * c + extra) * e + (8 * r if op == "cross_entropy" else 0), "flops": ops * r * c}
    if op == "rotary_embedding":
        n = case["batch"] * case["heads"] * case["seq"] * case["head_dim"]
        return {"bytes": (2 * n + case["seq"] * case["head_dim"]) * e, "flops": 3 * n}
    if op == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (m * k + k * n + m * n) * e, "flops": 2 * m * n * k}
    if op == "fused_mlp":
        m, d, h = case["rows"], case["dim"], case["hidden"]
        return {"bytes": (2 * m * d + 3 * d * h) * e, "flops": 6 * m * d * h}
    if op == "flash_attention":
        b, h, sq, sk, d = case["batch"], case["heads"], case["seq_q"], case["seq_k"], case["head_dim"]
        pairs = sq * (sq + 1) // 2 if case["causal"] else sq * sk
        return {"bytes": 2 * b * d * (h * sq + case["kv_heads"] * sk) * e, "flops": 4 * b * h * d * pairs}
    b, t, c = case["batch"], case["seq"], GPT2_WIDTH
    block = 12 * c * c
    return {"bytes": (GPT2_LAYERS * block + GPT2_VOCAB * c + b * t * GPT2_VOCAB) * e,
            "flops": 2 * b * t * (GPT2_LAYERS * block + GPT2_VOCAB * c) + GPT2_LAYERS * 2 * b * t * (t + 1) * c}


# Largest relative error of one rounding to the type.
_UNIT = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8, "f32": 2.0 ** -24}
# (2-norm, largest element) of the error in those units, about four times what the library's results
# show against 64 bits over 120 drawn cases of all sizes: one rounding of an exact value gives 0.43
# in the 2-norm and 1 at most. RMSNorm rounds four times and RoPE three, as tensor ops do; the MLP
# rounds gate, up, their product and the output; attention rounds P, and the early rows of a causal
# mask are far larger than the root mean square; the model carries roundings through twelve layers.
_UNITS = {"rmsnorm": (4, 12), "layernorm": (2, 5), "softmax": (2, 5), "cross_entropy": (4, 4),
          "rotary_embedding": (2.5, 16), "reduce": (2, 5), "matmul": (2, 5), "fused_mlp": (4, 22),
          "flash_attention": (2.5, 64), "gpt2": (11, 72)}
_UNITS_F32 = {"softmax": (8, 40), "matmul": (8, 40), "fused_mlp": (12, 60)}  # sums of 32-bit products


def tolerance(case: dict) -> dict:
    op, dtype = case["op"], case["dtype"]
    rel, most = _UNITS_F32.get(op, _UNITS[op]) if dtype == "f32" else _UNITS[op]
    if dtype == "f32" and op not in _UNITS_F32:
        rel, most = max(rel, 6), max(most, 24)
    return {"rel": rel * _UNIT[dtype], "max": most * _UNIT[dtype]}
