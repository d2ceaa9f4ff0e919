"""The work a program using this package has it do, as measurable cases.

Each case is a plain dict: ``kind`` names the path, the rest its sizes and
options. ``prepare`` makes what such a program holds before the call (inputs,
weights, a workspace it keeps), ``run`` is one pass through the public entry
points, ``work`` the bytes and operations the path cannot do without, ``exact``
the same result in float64 with plain torch.

Kinds:

* ``lora``       one LoRA projection, forward only (inference);
* ``lora_train`` the same projection forward and backward;
* ``block``      a whole Llama-shaped block forward (attention and MLP);
* ``attention``  the causal attention products and their softmax;
* ``paged``      one decode step of attention over a paged KV cache;
* ``norm``       the residual add and RMSNorm in front of a layer;
* ``probs``      softmax over vocabulary logits, to fp32 probabilities;
* ``weights``    block-wise INT8 quantisation of a weight and back.
"""

from __future__ import annotations

import math

import torch

import cuda_force_amd as cf
from cuda_force_amd import _lib, ops
from cuda_force_amd.transformer_block import BlockConfig, LlamaBlock

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_SIZE = {"bf16": 2, "f16": 2, "f32": 4}


def listed() -> list[dict]:
    return [
        # Token generation for a few sequences: one attention projection per
        # step, a handful of rows against the whole weight.
        {"name": "lora_decode", "kind": "lora", "dtype": "bf16", "m": 4, "k": 4096, "n": 4096, "rank": 16, "alpha": 32},
        # One user's prompt through an MLP up-projection: ragged row count.
        {"name": "lora_prompt", "kind": "lora", "dtype": "bf16", "m": 333, "k": 4096, "n": 11008, "rank": 16,
         "alpha": 32},
        # The benchmark's large projection: a full prefill batch.
        {"name": "lora_prefill", "kind": "lora", "dtype": "bf16", "m": 8192, "k": 4096, "n": 4096, "rank": 16,
         "alpha": 32},
        # A fine-tuning step of one adapted layer inside a stack (its input
        # needs a gradient too), 8 sequences of 512 tokens.
        {"name": "lora_train", "kind": "lora_train", "dtype": "bf16", "m": 4096, "k": 4096, "n": 4096, "rank": 16,
         "alpha": 32},
        # The same with a larger adapter and a ragged batch of tokens.
        {"name": "lora_train_rank64", "kind": "lora_train", "dtype": "bf16", "m": 2000, "k": 4096, "n": 4096,
         "rank": 64, "alpha": 16},
        # Full-precision fine-tuning at the reference's benchmark shape.
        {"name": "lora_train_fp32", "kind": "lora_train", "dtype": "f32", "m": 128, "k": 4096, "n": 4096, "rank": 16,
         "alpha": 16},
        # One whole 7B-shaped block over 8 x 512 tokens.
        {"name": "block", "kind": "block", "hidden": 4096, "heads": 32, "inner": 11008, "rank": 16, "batch": 8,
         "seq": 512},
        # Attention of one longer prompt.
        {"name": "attention_2048", "kind": "attention", "batch": 1, "seq": 2048, "heads": 32, "dim": 128},
        # One decode step over a paged cache: 64 sequences of mixed length,
        # grouped-query heads.
        {"name": "paged_decode", "kind": "paged", "dtype": "bf16", "sequences": 64, "context": 1024, "heads": 32,
         "kv_heads": 8, "dim": 128, "block": 16},
        # The norm in front of a layer while generating: the smallest call.
        {"name": "norm_decode", "kind": "norm", "dtype": "bf16", "rows": 4, "hidden": 4096},
        # Next-token probabilities of a batch of positions.
        {"name": "vocab_probs", "kind": "probs", "dtype": "bf16", "rows": 257, "cols": 32000},
        # Quantising and restoring one 7B MLP weight.
        {"name": "weight_int8", "kind": "weights", "dtype": "bf16", "rows": 11008, "cols": 4096},
    ]


def _log(rng, low: int, high: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _width(rng, low: int, high: int) -> int:
    """A layer width: a common one, or any multiple of 8 in the range."""
    common = [w for w in (256, 512, 688, 1024, 2048, 4096, 5120, 8192, 11008) if low <= w <= high]
    return rng.choice(common) if rng.random() < 0.6 else 8 * _log(rng, low // 8, high // 8)


def draw(rng) -> dict:
    kind = rng.choice(["lora", "lora", "lora", "lora_train", "lora_train", "lora_train", "block", "attention",
                       "paged", "norm", "probs", "weights"])
    if kind == "lora":
        return {"kind": kind, "dtype": "f32" if rng.random() < 0.15 else "bf16", "m": _log(rng, 1, 6000),
                "k": _width(rng, 256, 11008), "n": _width(rng, 256, 11008), "rank": rng.choice([4, 8, 16, 16, 32, 64]),
                "alpha": rng.choice([16, 32])}
    if kind == "lora_train":
        fp32 = rng.random() < 0.2
        return {"kind": kind, "dtype": "f32" if fp32 else "bf16", "m": _log(rng, 16, 1024 if fp32 else 5000),
                "k": _width(rng, 256, 4096), "n": _width(rng, 256, 4096 if fp32 else 11008),
                "rank": rng.choice([4, 8, 16, 16, 32, 64]), "alpha": rng.choice([16, 32])}
    if kind == "block":
        hidden, heads, inner = rng.choice([(256, 4, 688), (512, 8, 1024), (1024, 16, 2752), (2048, 16, 5504)])
        return {"kind": kind, "hidden": hidden, "heads": heads, "inner": inner, "rank": rng.choice([8, 16]),
                "batch": rng.randint(1, 8), "seq": 8 * rng.randint(4, 96)}
    if kind == "attention":
        seq = 8 * _log(rng, 8, 256)
        return {"kind": kind, "batch": rng.randint(1, max(1, min(8, 2048 // seq))), "seq": seq,
                "heads": rng.choice([8, 16, 32]), "dim": rng.choice([64, 128])}
    if kind == "paged":
        heads, kv_heads = rng.choice([(32, 32), (32, 8), (64, 8), (16, 8)])
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f32"]), "sequences": _log(rng, 1, 128),
                "context": _log(rng, 32, 1024), "heads": heads, "kv_heads": kv_heads, "dim": rng.choice([64, 128]),
                "block": rng.choice([16, 32])}
    if kind == "norm":
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "rows": _log(rng, 1, 8192),
                "hidden": _width(rng, 256, 8192)}
    if kind == "probs":
        return {"kind": kind, "dtype": rng.choice(["bf16", "f16", "f32"]), "rows": _log(rng, 1, 1024),
                "cols": rng.choice([32000, 32001, 50257, 65536, _log(rng, 1000, 70000)])}
    return {"kind": kind, "dtype": rng.choice(["bf16", "f32"]), "rows": _log(rng, 64, 11008),
            "cols": _log(rng, 64, 4096)}


# ---------------------------------------------------------------------------
# Inputs.
# ---------------------------------------------------------------------------


class _Inputs:
    """Seeded normal tensors on the GPU."""

    def __init__(self, seed: int) -> None:
        self.gen = torch.Generator(device="cuda").manual_seed(1_000_003 * (seed % 1_000_003) + 17)

    def normal(self, *shape: int, std: float = 1.0, dtype: torch.dtype = torch.float32) -> torch.Tensor:
        return (std * torch.randn(*shape, generator=self.gen, device="cuda")).to(dtype)


def prepare(case: dict, seed: int) -> dict:
    return _PREPARE[case["kind"]](case, _Inputs(seed))


def _prepare_lora(case: dict, inputs: _Inputs) -> dict:
    dtype = _DTYPES[case["dtype"]]
    m, k, n, r = case["m"], case["k"], case["n"], case["rank"]
    return {
        "kind": case["kind"],
        "x": inputs.normal(m, k, dtype=dtype),
        "w": inputs.normal(k, n, std=0.02, dtype=dtype),
        "a": inputs.normal(k, r, std=1 / 64, dtype=dtype),
        "b": inputs.normal(r, n, std=0.02, dtype=dtype),
        "scale": case["alpha"] / r,
    }


def _prepare_lora_train(case: dict, inputs: _Inputs) -> dict:
    state = _prepare_lora(case, inputs)
    state["grad_y"] = inputs.normal(case["m"], case["n"], dtype=_DTYPES[case["dtype"]])
    for name in ("x", "a", "b"):  # the base weight is frozen
        state[name].requires_grad_(True)
    return state


def _prepare_block(case: dict, inputs: _Inputs) -> dict:
    config = BlockConfig(hidden=case["hidden"], heads=case["heads"], intermediate=case["inner"], rank=case["rank"],
                         alpha=2.0 * case["rank"])
    block = LlamaBlock(config, "cuda", torch.bfloat16, inputs.gen)
    shape = (case["batch"], case["seq"], case["hidden"])
    return {"kind": "block", "block": block, "x": inputs.normal(*shape, dtype=torch.bfloat16),
            "residual": inputs.normal(*shape, dtype=torch.bfloat16)}


def _prepare_attention(case: dict, inputs: _Inputs) -> dict:
    shape = (case["batch"], case["seq"], case["heads"] * case["dim"])
    q, k, v = (inputs.normal(*shape, dtype=torch.bfloat16) for _ in range(3))
    return {"kind": "attention", "q": q, "k": k, "v": v, "heads": case["heads"], "seq": case["seq"],
            "scale": 1.0 / math.sqrt(case["dim"])}


def _contexts(case: dict) -> list[int]:
    """Mixed lengths, from a quarter of the longest up."""
    s, longest = case["sequences"], case["context"]
    low = max(1, longest // 4)
    return [longest - (i * 7919) % (longest - low + 1) for i in range(s)]


def _prepare_paged(case: dict, inputs: _Inputs) -> dict:
    dtype = _DTYPES[case["dtype"]]
    s, h, kvh, d, bs = case["sequences"], case["heads"], case["kv_heads"], case["dim"], case["block"]
    contexts = _contexts(case)
    max_blocks = (max(contexts) + bs - 1) // bs
    total = s * max_blocks
    order = torch.randperm(total, generator=inputs.gen, device="cuda").to(torch.int32)
    lib = _lib.load()
    nbytes = lib.cf_paged_attention_workspace_bytes(s, h, kvh, d, bs, max_blocks)
    return {
        "kind": "paged",
        "q": inputs.normal(s, h, d, dtype=dtype),
        "k": inputs.normal(total, bs, kvh, d, dtype=dtype),
        "v": inputs.normal(total, bs, kvh, d, dtype=dtype),
        "tables": order.view(s, max_blocks).contiguous(),
        "contexts": torch.tensor(contexts, dtype=torch.int32, device="cuda"),
        "out": torch.zeros(s, h, d, dtype=dtype, device="cuda"),
        "workspace": torch.zeros(max(nbytes, 1), dtype=torch.uint8, device="cuda"),
        "nbytes": nbytes,
        "dims": (s, h, kvh, d, bs, max_blocks),
        "code": _lib.dtype_code(dtype),
        "scale": 1.0 / math.sqrt(d),
    }


def _prepare_norm(case: dict, inputs: _Inputs) -> dict:
    dtype = _DTYPES[case["dtype"]]
    rows, hidden = case["rows"], case["hidden"]
    return {"kind": "norm", "x": inputs.normal(rows, hidden, dtype=dtype),
            "residual": inputs.normal(rows, hidden, dtype=dtype),
            "weight": (1 + inputs.normal(hidden, std=0.02)).to(dtype)}


def _prepare_probs(case: dict, inputs: _Inputs) -> dict:
    return {"kind": "probs", "logits": inputs.normal(case["rows"], case["cols"], std=2.0, dtype=_DTYPES[case["dtype"]])}


def _prepare_weights(case: dict, inputs: _Inputs) -> dict:
    rows, cols = case["rows"], case["cols"]
    w = inputs.normal(rows, cols, std=0.02)
    flat = w.view(-1)
    outliers = torch.randint(0, flat.numel(), (max(1, flat.numel() // 1000),), generator=inputs.gen, device="cuda")
    flat[outliers] = flat[outliers] * 50.0
    return {"kind": "weights", "w": w.to(_DTYPES[case["dtype"]])}


_PREPARE = {"lora": _prepare_lora, "lora_train": _prepare_lora_train, "block": _prepare_block,
            "attention": _prepare_attention, "paged": _prepare_paged, "norm": _prepare_norm,
            "probs": _prepare_probs, "weights": _prepare_weights}


# ---------------------------------------------------------------------------
# One pass.
# ---------------------------------------------------------------------------


def run(state: dict):
    return _RUN[state["kind"]](state)


def _run_lora(s: dict):
    return cf.lora_linear(s["x"], s["w"], s["a"], s["b"], s["scale"])


def _run_lora_train(s: dict):
    y = cf.lora_linear(s["x"], s["w"], s["a"], s["b"], s["scale"])
    grad_x, grad_a, grad_b = torch.autograd.grad(y, (s["x"], s["a"], s["b"]), s["grad_y"])
    return {"y": y.detach(), "grad_x": grad_x, "grad_a": grad_a, "grad_b": grad_b}


def _run_block(s: dict):
    out, residual = s["block"].forward(s["x"], s["residual"])
    return {"out": out, "residual": residual}


def _run_attention(s: dict):
    scores = ops.attention_scores_causal(s["q"], s["k"], s["heads"])
    weights = cf.softmax_scaled(scores.view(-1, s["seq"]), s["scale"], s["seq"]).view_as(scores)
    return ops.attention_pv_causal(weights, s["v"], s["heads"])


def _run_paged(s: dict):
    lib = _lib.load()
    _lib.check(lib.cf_paged_attention(
        s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["tables"].data_ptr(), s["contexts"].data_ptr(),
        s["out"].data_ptr(), s["code"], *s["dims"], s["scale"], s["workspace"].data_ptr() if s["nbytes"] else None,
        s["nbytes"], torch.cuda.current_stream().cuda_stream))
    return s["out"]


def _run_norm(s: dict):
    normed, summed = cf.fused_residual_rmsnorm(s["x"], s["residual"], s["weight"], 1e-6)
    return {"normed": normed, "summed": summed}


def _run_probs(s: dict):
    return cf.softmax_as(s["logits"], torch.float32)


def _run_weights(s: dict):
    codes, scales = cf.quantize_int8(s["w"])
    return {"codes": codes, "scales": scales, "restored": cf.dequantize_int8(codes, scales, s["w"].dtype)}


_RUN = {"lora": _run_lora, "lora_train": _run_lora_train, "block": _run_block, "attention": _run_attention,
        "paged": _run_paged, "norm": _run_norm, "probs": _run_probs, "weights": _run_weights}


# ---------------------------------------------------------------------------
# What a pass cannot do without: inputs read once, outputs written once.
# ---------------------------------------------------------------------------


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("lora", "lora_train"):
        e = _SIZE[case["dtype"]]
        m, k, n, r = case["m"], case["k"], case["n"], case["rank"]
        inputs = m * k + k * n + k * r + r * n
        flops = 2 * m * k * n + 2 * m * k * r + 2 * m * r * n
        if kind == "lora":
            return {"bytes": e * (inputs + m * n), "flops": flops}
        # grad_y read; y, grad_x, grad_a, grad_b written.
        total = inputs + m * n + (m * n + m * k + k * r + r * n)
        return {"bytes": e * total, "flops": 2 * flops + 2 * m * k * r + 2 * m * r * n}
    if kind == "block":
        h, i, r, b, s = case["hidden"], case["inner"], case["rank"], case["batch"], case["seq"]
        t = b * s
        widths = [(h, h)] * 4 + [(h, i)] * 2 + [(i, h)]
        weights = sum(p * q + r * (p + q) for p, q in widths) + 2 * h
        attention = 2 * 2 * b * h * s * (s + 1) // 2  # the causal half of both products
        return {"bytes": 2 * (weights + 4 * t * h),
                "flops": sum(2 * t * (p * q + r * (p + q)) for p, q in widths) + attention}
    if kind == "attention":
        rows = case["batch"] * case["seq"] * case["heads"] * case["dim"]
        half = case["batch"] * case["heads"] * case["seq"] * (case["seq"] + 1) // 2
        # The scores and the whole probability matrix are results of the
        # path's own entry points: written once and read once (causal half).
        full = case["batch"] * case["heads"] * case["seq"] * case["seq"]
        return {"bytes": 2 * (4 * rows + 3 * half + full), "flops": 4 * half * case["dim"]}
    if kind == "paged":
        e = _SIZE[case["dtype"]]
        tokens = sum(_contexts(case))
        rows = case["sequences"] * case["heads"] * case["dim"]
        return {"bytes": e * (2 * tokens * case["kv_heads"] * case["dim"] + 2 * rows),
                "flops": 4 * tokens * case["heads"] * case["dim"]}
    if kind == "norm":
        e = _SIZE[case["dtype"]]
        return {"bytes": e * (4 * case["rows"] * case["hidden"] + case["hidden"]),
                "flops": 5 * case["rows"] * case["hidden"]}
    if kind == "probs":
        return {"bytes": (_SIZE[case["dtype"]] + 4) * case["rows"] * case["cols"],
                "flops": 4 * case["rows"] * case["cols"]}
    count = case["rows"] * case["cols"]
    return {"bytes": int(count * (2 * _SIZE[case["dtype"]] + 2 + 2 * 4 / 64)), "flops": 4 * count}


# Relative error (2-norm) of the results against float64, measured on the
# listed cases and drawn ones, times about four. Measured: one bf16 rounding
# 1.7e-3 (lora), gradients and the normed row 2.4e-3 (an intermediate is
# rounded too), attention 3.6e-3 (rounded probabilities), paged 3.0e-3, a
# whole block 6.6e-3; fp32 LoRA 4.5e-6 (products of bf16 high and low parts),
# fp32 norm 6e-8, fp32 probabilities 7.5e-8.
def tolerance(case: dict):
    kind = case["kind"]
    if kind == "weights":
        return "exact"
    if kind == "lora":
        return {"rel": 2e-5 if case["dtype"] == "f32" else 7e-3}
    if kind == "lora_train":
        return {"rel": 2e-5 if case["dtype"] == "f32" else 1e-2}
    if kind == "block":
        return {"rel": 2.6e-2}
    if kind == "attention":
        return {"rel": 1.4e-2}
    if kind == "paged":
        return {"rel": 1e-5 if case["dtype"] == "f32" else 1.2e-2}
    if kind == "norm":
        return {"rel": {"f32": 5e-7, "f16": 1.5e-3, "bf16": 1e-2}[case["dtype"]]}
    return {"rel": 5e-7}


# ---------------------------------------------------------------------------
# The same results in float64.
# ---------------------------------------------------------------------------


def exact(case: dict, seed: int):
    return _EXACT[case["kind"]](prepare(case, seed))


def _exact_lora(s: dict):
    x, w, a, b = (s[name].detach().double() for name in ("x", "w", "a", "b"))
    return x @ w + s["scale"] * ((x @ a) @ b)


def _exact_lora_train(s: dict):
    x, w, a, b, dy = (s[name].detach().double() for name in ("x", "w", "a", "b", "grad_y"))
    scale = s["scale"]
    g = dy @ b.t().contiguous()
    return {"y": x @ w + scale * ((x @ a) @ b), "grad_x": dy @ w.t().contiguous() + scale * (g @ a.t().contiguous()),
            "grad_a": scale * (x.t().contiguous() @ g), "grad_b": scale * ((x @ a).t().contiguous() @ dy)}


def _causal_attention(q, k, v, heads: int, scale: float):
    """[batch, seq, heads * dim] in float64, one batch entry at a time."""
    batch, seq, hidden = q.shape
    mask = torch.triu(torch.full((seq, seq), float("-inf"), dtype=torch.float64, device=q.device), 1)
    out = torch.empty_like(q)
    for i in range(batch):
        qh, kh, vh = (t[i].view(seq, heads, -1).transpose(0, 1).contiguous() for t in (q, k, v))
        p = torch.softmax(scale * torch.bmm(qh, kh.transpose(1, 2).contiguous()) + mask, dim=-1)
        out[i] = torch.bmm(p, vh).transpose(0, 1).reshape(seq, hidden)
    return out


def _exact_attention(s: dict):
    return _causal_attention(s["q"].double(), s["k"].double(), s["v"].double(), s["heads"], s["scale"])


def _exact_block(s: dict):
    block = s["block"]
    c = block.config

    def norm(t, weight):
        return t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + c.eps) * weight.double()

    def project(p, t):
        return t @ p.w.double() + p.scale * ((t @ p.a.double()) @ p.b.double())

    residual = s["x"].double() + s["residual"].double()
    normed = norm(residual, block.attention_norm)
    q, k, v = (project(p, normed) for p in (block.q, block.k, block.v))
    residual = residual + project(block.o, _causal_attention(q, k, v, c.heads, 1.0 / math.sqrt(c.head_dim)))
    normed = norm(residual, block.ffn_norm)
    out = project(block.down, torch.nn.functional.silu(project(block.gate, normed)) * project(block.up, normed))
    return {"out": out, "residual": residual}


def _exact_paged(s: dict):
    sequences, heads, kv_heads, dim, block, _ = s["dims"]
    out = torch.empty(sequences, heads, dim, dtype=torch.float64, device="cuda")
    group = heads // kv_heads
    for i, context in enumerate(s["contexts"].tolist()):
        blocks = s["tables"][i, : (context + block - 1) // block].long()
        keys, values = (s[name][blocks].reshape(-1, kv_heads, dim)[:context].double().transpose(0, 1)
                        .repeat_interleave(group, dim=0).contiguous() for name in ("k", "v"))
        scores = s["scale"] * torch.bmm(keys, s["q"][i].double().unsqueeze(2).contiguous()).squeeze(2)
        out[i] = torch.bmm(torch.softmax(scores, dim=-1).unsqueeze(1), values).squeeze(1)
    return out


def _exact_norm(s: dict):
    summed = s["x"].double() + s["residual"].double()
    inverse = torch.rsqrt(summed.pow(2).mean(-1, keepdim=True) + 1e-6)
    return {"normed": summed * inverse * s["weight"].double(), "summed": summed}


def _exact_probs(s: dict):
    return torch.softmax(s["logits"].double(), dim=-1)


def _exact_weights(s: dict):
    """The scales alone: codes and restored values are whole numbers and their
    products with a scale, compared bit for bit."""
    flat = s["w"].double().view(-1)
    padded = torch.nn.functional.pad(flat, (0, -flat.numel() % cf.QUANT_BLOCK_SIZE))
    return {"codes": None, "scales": padded.view(-1, cf.QUANT_BLOCK_SIZE).abs().amax(1) / 127.0, "restored": None}


_EXACT = {"lora": _exact_lora, "lora_train": _exact_lora_train, "block": _exact_block, "attention": _exact_attention,
          "paged": _exact_paged, "norm": _exact_norm, "probs": _exact_probs, "weights": _exact_weights}
