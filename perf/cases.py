"""Calls that a program serving a GGUF model makes of this framework, as measurable cases.

Every case is one call (or the calls of one decoder layer) through the public entry points of
``vllm_gguf_plugin_prism_amd.dispatch``, with packed weights resident on the GPU and fresh activations.  There are four
kinds:

``linear``  one linear layer: ``fused_mul_mat_gguf`` on ``m`` rows of activations (1 row: decode of one sequence; a few:
            decode of a batch; tens to thousands: prefill), any of the 19 formats
``layer``   the linear layers of one decoder layer, as a decode step calls them one after the other: merged q/k/v,
            output, merged gate/up, down; formats as a quantization recipe mixes them (v and down in more bits)
``moe``     a mixture-of-experts layer: ``fused_moe_gguf`` on ``m`` tokens routed to ``top_k`` of ``experts``
``embed``   the embedding lookup of ``m`` token ids from a packed table
"""
from __future__ import annotations

import math

import torch

from vllm_gguf_plugin_prism_amd import dispatch, synth

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}

# ggml name -> (type id, offsets of the fp16 super-scales in a block, what the standard deviation of a weight is when
# the first of them is 1 and the other fields are uniformly random, the second one over the first)
FORMATS = {
    "Q4_0": (2, (0,), 4.6, 0), "Q4_1": (3, (0, 2), 4.6, -7.5), "Q5_0": (6, (0,), 9.2, 0), "Q5_1": (7, (0, 2), 9.2, -15.5),
    "Q8_0": (8, (0,), 74, 0), "Q2_K": (10, (80, 82), 13, 1.5), "Q3_K": (11, (108,), 43, 0), "Q4_K": (12, (0, 2), 320, 7.5),
    "Q5_K": (13, (0, 2), 640, 15.5), "Q6_K": (14, (208,), 1370, 0), "IQ2_XXS": (16, (0,), 60, 0), "IQ2_XS": (17, (0,), 60, 0),
    "IQ3_XXS": (18, (0,), 130, 0), "IQ1_S": (19, (0,), 8, 0), "IQ4_NL": (20, (0,), 70, 0), "IQ3_S": (21, (0,), 150, 0),
    "IQ2_S": (22, (0,), 60, 0), "IQ4_XS": (23, (0,), 1300, 0), "IQ1_M": (29, (), 8, 0),
}
MATRIX_FORMATS = ("Q4_0", "Q4_1", "Q5_0", "Q5_1", "Q8_0", "Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K")
# recipe -> (most tensors of a layer, its v and down projections)
RECIPES = {"Q4_K_M": ("Q4_K", "Q6_K"), "Q5_K_M": ("Q5_K", "Q6_K"), "Q3_K_M": ("Q3_K", "Q5_K"), "Q4_0": ("Q4_0", "Q4_0"),
           "Q8_0": ("Q8_0", "Q8_0"), "Q6_K": ("Q6_K", "Q6_K"), "IQ4_XS": ("IQ4_XS", "Q5_K")}

MOST_FLOPS = 2 * 1531 * 4096 * 14336  # the largest listed case
MOST_MOE_FLOPS = 60e9


def listed() -> list[dict]:
    return [
        # a small model's projection, one sequence: 3 MB of weights, so launch and host path are what it costs
        {"name": "linear_q8_0_1row_small", "kind": "linear", "format": "Q8_0", "n": 3072, "k": 1024, "m": 1, "dtype": "fp16"},
        # one decode step of one sequence through a layer of an 8B-class model in the most common mixed recipe
        {"name": "layer_q4_k_m_1row", "kind": "layer", "recipe": "Q4_K_M", "hidden": 4096, "kv": 1024, "inner": 14336, "m": 1, "dtype": "fp16"},
        # the same layer for a batch of 12 sequences
        {"name": "layer_q4_k_m_12rows", "kind": "layer", "recipe": "Q4_K_M", "hidden": 4096, "kv": 1024, "inner": 14336, "m": 12, "dtype": "bf16"},
        # a codebook format, decode of one sequence
        {"name": "linear_iq2_xxs_1row", "kind": "linear", "format": "IQ2_XXS", "n": 17408, "k": 5120, "m": 1, "dtype": "fp16"},
        # a codebook format on a short prompt: no tile kernel in the reference's policy, weights are dequantized first
        {"name": "linear_iq4_xs_256rows", "kind": "linear", "format": "IQ4_XS", "n": 5120, "k": 5120, "m": 256, "dtype": "bf16"},
        # a short, odd-sized prompt (or a large decode batch)
        {"name": "linear_q8_0_77rows", "kind": "linear", "format": "Q8_0", "n": 14336, "k": 4096, "m": 77, "dtype": "bf16"},
        # a prompt of 512 tokens: the integer GEMM on the format with a scale for every 16 weights
        {"name": "linear_q6_k_512rows", "kind": "linear", "format": "Q6_K", "n": 18944, "k": 3584, "m": 512, "dtype": "fp16"},
        # a long prompt's ragged last chunk: the largest call
        {"name": "linear_q4_k_1531rows", "kind": "linear", "format": "Q4_K", "n": 4096, "k": 14336, "m": 1531, "dtype": "bf16"},
        # mixture of experts, decode of one sequence
        {"name": "moe_q4_0_1token", "kind": "moe", "format": "Q4_0", "format2": "Q4_0", "experts": 64, "top_k": 8, "hidden": 2048, "inner": 1024, "m": 1, "dtype": "fp16"},
        # the same for a batch: every expert is hit, by a few tokens each
        {"name": "moe_q4_0_64tokens", "kind": "moe", "format": "Q4_0", "format2": "Q4_0", "experts": 64, "top_k": 8, "hidden": 2048, "inner": 1024, "m": 64, "dtype": "fp16"},
        # many small experts in a mixed recipe, a prompt
        {"name": "moe_q4_k_q6_k_300tokens", "kind": "moe", "format": "Q4_K", "format2": "Q6_K", "experts": 128, "top_k": 8, "hidden": 2048, "inner": 768, "m": 300, "dtype": "bf16"},
        # the embedding rows of a prompt
        {"name": "embed_q6_k_211ids", "kind": "embed", "format": "Q6_K", "n": 128000, "k": 4096, "m": 211, "dtype": "bf16"},
    ]


def _spread(rng, lo: int, hi: int, step: int = 1) -> int:
    """A multiple of ``step`` between ``lo`` and ``hi``, uniform in its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, round(v / step) * step))


def draw(rng) -> dict:
    kind = rng.choice(("linear", "linear", "linear", "linear", "layer", "layer", "moe", "moe", "moe", "embed"))
    case = {"kind": kind, "dtype": rng.choice(("fp16", "bf16"))}
    while True:
        if kind == "linear":
            fmt = rng.choice(MATRIX_FORMATS if rng.random() < 0.6 else tuple(FORMATS))
            step = 256 if synth.QUANT_SIZES[FORMATS[fmt][0]][0] == 256 else 32
            case.update(format=fmt, n=_spread(rng, 512, 28672, 16), k=_spread(rng, 512, 18944, step), m=_spread(rng, 1, 2048))
        elif kind == "layer":
            hidden = _spread(rng, 1024, 8192, 256)
            case.update(recipe=rng.choice(tuple(RECIPES)), hidden=hidden, kv=rng.choice((256, 512, 1024)),
                        inner=_spread(rng, 2 * hidden, 4 * hidden, 256), m=_spread(rng, 1, 64))
        elif kind == "moe":
            fmt = rng.choice(("Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"))
            experts = rng.choice((8, 16, 32, 64, 128))
            case.update(format=fmt, format2="Q6_K" if fmt in ("Q4_K", "Q5_K") and rng.random() < 0.6 else fmt, experts=experts,
                        top_k=2 if experts <= 16 else rng.choice((4, 6, 8)), hidden=_spread(rng, 1024, 4096, 256),
                        inner=_spread(rng, 512, 8192, 256), m=_spread(rng, 1, 1024))
        else:
            case.update(format=rng.choice(("Q4_K", "Q6_K", "Q8_0")), n=_spread(rng, 32000, 152000, 64), k=_spread(rng, 1024, 8192, 256),
                        m=_spread(rng, 1, 2048))
        w = work(case)
        if w["flops"] <= (MOST_MOE_FLOPS if kind == "moe" else MOST_FLOPS) and _weight_bytes(case) <= 600e6:
            return case


# ---------------------------------------------------------------------------------------------------------------- inputs


def _row_bytes(fmt: str, k: int) -> int:
    qk, size = synth.QUANT_SIZES[FORMATS[fmt][0]]
    return k // qk * size


def _pack(gen, fmt: str, n: int, k: int) -> torch.Tensor:
    """Packed rows ``uint8[n, row bytes]``: random codes and scales, super-scales such that the weights spread as 0.02."""
    type_id, at, unit, ratio = FORMATS[fmt]
    qk, size = synth.QUANT_SIZES[type_id]
    raw = torch.randint(0, 256, (n * k // qk, size), dtype=torch.uint8, device="cuda", generator=gen)
    d = (0.02 / unit * (0.5 + torch.rand(raw.shape[0], device="cuda", generator=gen))).to(torch.float16)
    for i, o in enumerate(at):
        raw[:, o:o + 2] = (d if i == 0 else (d.float() * ratio).to(torch.float16)).view(torch.uint8).reshape(-1, 2)
    if fmt == "IQ1_M":  # its super-scale lies in the top four bits of four 16-bit words
        bits = d.view(torch.int16).to(torch.int32)
        for i in range(4):
            raw[:, 49 + 2 * i] = ((raw[:, 49 + 2 * i].to(torch.int32) & 15) | ((bits >> (4 * i)) & 15) << 4).to(torch.uint8)
    return raw.reshape(n, -1)


def _activations(gen, m: int, k: int, dtype) -> torch.Tensor:
    """Hidden states: unit variance, with the few channels of large values that transformers have."""
    channel = 1 + 7 * (torch.rand(k, device="cuda", generator=gen) > 0.995).float()
    return (torch.randn(m, k, device="cuda", generator=gen) * channel).to(dtype)


def _layer_parts(case):
    """(rows, columns, format) of every packed tensor of a decoder layer, the merged q/k/v as three."""
    most, more = RECIPES[case["recipe"]]
    h, kv, inner = case["hidden"], case["kv"], case["inner"]
    return [(h, h, most), (kv, h, most), (kv, h, more), (h, h, most), (2 * inner, h, most), (h, inner, more)]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, m, kind = DTYPES[case["dtype"]], case["m"], case["kind"]
    if kind == "linear":
        return {"kind": kind, "w": _pack(gen, case["format"], case["n"], case["k"]), "type": FORMATS[case["format"]][0],
                "x": _activations(gen, m, case["k"], dtype)}
    if kind == "embed":
        return {"kind": kind, "w": _pack(gen, case["format"], case["n"], case["k"]), "type": FORMATS[case["format"]][0],
                "ids": torch.randint(0, case["n"], (m,), device="cuda", generator=gen), "hidden": case["k"], "dtype": dtype}
    if kind == "moe":
        e, h, inner = case["experts"], case["hidden"], case["inner"]
        # experts are not hit evenly
        logits = torch.randn(m, e, device="cuda", generator=gen) + 0.5 * torch.randn(e, device="cuda", generator=gen)
        weights, ids = torch.topk(torch.softmax(logits, 1), case["top_k"])
        return {"kind": kind, "w1": _pack(gen, case["format"], e * 2 * inner, h).reshape(e, 2 * inner, -1),
                "w2": _pack(gen, case["format2"], e * h, inner).reshape(e, h, -1), "weights": weights,
                "ids": ids.to(torch.int32), "x": _activations(gen, m, h, dtype), "type": FORMATS[case["format"]][0],
                "type2": FORMATS[case["format2"]][0]}
    parts = [(_pack(gen, fmt, n, k), FORMATS[fmt][0]) for n, k, fmt in _layer_parts(case)]
    (q, most), (k_, _), (v, more), o, gate_up, down = parts
    # the merged tensor is as wide as its widest shard, the others' rows are padded
    width = max(t.shape[1] for t in (q, k_, v))
    qkv = torch.zeros(q.shape[0] + 2 * k_.shape[0], width, dtype=torch.uint8, device="cuda")
    shards, start = {}, 0
    for i, t in zip("qkv", (q, k_, v)):
        qkv[start:start + t.shape[0], :t.shape[1]] = t
        shards[i] = (start, start + t.shape[0], t.shape[1])
        start += t.shape[0]
    x, h = _activations(gen, m, case["hidden"], dtype), _activations(gen, m, case["inner"], dtype)
    return {"kind": kind, "qkv": qkv, "shards": shards, "types": {"q": most, "k": most, "v": more},
            "rest": [(*o, x, ()), (*gate_up, x, ("gate", "up")), (*down, h, ())], "x": x,
            "bias": _activations(gen, 1, qkv.shape[0], dtype).reshape(-1)}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return dispatch.fused_mul_mat_gguf(state["x"], state["w"], state["type"])
    if kind == "embed":
        return dispatch.apply_gguf_embedding(state["ids"], state["w"], state["type"], state["hidden"], state["dtype"])
    if kind == "moe":
        return dispatch.fused_moe_gguf(state["x"], state["w1"], state["w2"], state["weights"], state["ids"], state["type"], state["type2"], "silu")
    y = [dispatch.apply_linear(state["x"], state["qkv"], state["types"]["q"], shard_ids=("q", "k", "v"), shard_offset_map=state["shards"],
                               shard_weight_types=state["types"], bias=state["bias"])]
    for w, type_id, x, shard_ids in state["rest"]:
        y.append(dispatch.apply_linear(x, w, type_id, shard_ids=shard_ids))
    return y


# ------------------------------------------------------------------------------------------------------------------ work


def _weight_bytes(case) -> float:
    """All packed weights of the case."""
    if case["kind"] == "moe":
        return case["experts"] * (2 * case["inner"] * _row_bytes(case["format"], case["hidden"]) + case["hidden"] * _row_bytes(case["format2"], case["inner"]))
    if case["kind"] == "layer":
        return sum(n * _row_bytes(fmt, k) for n, k, fmt in _layer_parts(case))
    return case["n"] * _row_bytes(case["format"], case["k"])


def work(case):
    """Packed weights that the call needs (each expert that is hit once, as many as uniform routing hits; the looked-up
    rows once), activations and results."""
    m, kind = case["m"], case["kind"]
    if kind == "linear":
        return {"bytes": _weight_bytes(case) + 2 * m * (case["k"] + case["n"]), "flops": 2 * m * case["n"] * case["k"]}
    if kind == "embed":
        return {"bytes": m * (_row_bytes(case["format"], case["k"]) + 2 * case["k"] + 8), "flops": 0}
    if kind == "moe":
        hit = 1 - (1 - case["top_k"] / case["experts"]) ** m
        return {"bytes": hit * _weight_bytes(case) + 4 * m * case["hidden"] + 8 * m * case["top_k"],
                "flops": 2 * m * case["top_k"] * 3 * case["inner"] * case["hidden"]}
    parts = _layer_parts(case)
    return {"bytes": _weight_bytes(case) + 2 * m * (case["hidden"] + case["inner"] + sum(n for n, _, _ in parts)),
            "flops": sum(2 * m * n * k for n, k, _ in parts)}


def tolerance(case):
    """Results are rounded to 16 bits once (the expert layer rounds between its products too); sums are 32-bit."""
    if case["kind"] == "embed":
        return "exact"
    return {"rel": 1e-3 if case["dtype"] == "fp16" else 6e-3}
