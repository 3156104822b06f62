"""Workloads the packed encoder path is measured on, each through a public entry point.

A case is a dict of plain values; its segment lengths follow from the case alone (``dist``,
``lo``, ``hi``, ``median``, ``n``, ``batch``), its tensors from the seed.

Kinds of call (``op``):

- ``attention``: ``varlen_attention`` over a packed batch. head_dim 64 calls are what a layer of
  the packed forward issues (q and k contiguous from the RoPE kernel, v a strided view of the
  packed projection); grouped-query calls have tensors of their own, with a sigmoid gate where
  the layer has one.
- ``prefixed``: ``varlen_attention`` with key segments of their own: rows that continue a cached
  prefix, from a single decoded token to a tail of some dozens.
- ``rope_attention``: ``ops.flash_attention_qkv_bshd``, RoPE and attention from the projection.
- ``layer``: ``forward.encoder_layer``, one ModernBERT layer with its norms, products and MLP.
- ``forward``: ``packed_forward``, the whole ModernBERT-base encoder.
"""

from __future__ import annotations

import math

import torch
from torch import nn

import packed_encoders_amd as pe
from packed_encoders_amd import forward, ops, workloads
from packed_encoders_amd.config import ModernBertParams

VOCAB = 50368
THETA = {True: 160000.0, False: 10000.0}  # RoPE base of global and local layers
HALF_WINDOW = 64
BASE = {"hidden": 768, "hq": 12, "mlp": 1152}
LARGE = {"hidden": 1024, "hq": 16, "mlp": 2624}


def listed() -> list[dict]:
    mha64 = {"op": "attention", "hq": 12, "hkv": 12, "d": 64, "window": -1, "causal": False, "gate": False}
    return [
        # an online search service's attention call: 32 short queries; launches and host time
        {"name": "queries_small", **mha64, "dist": "uniform", "n": 32, "lo": 16, "hi": 64, "batch": 1},
        # offline encoding of short queries: RoPE fused into the short-segment kernel
        {"name": "queries_rope_large", "op": "rope_attention", "hq": 12, "d": 64, "window": -1,
         "dist": "uniform", "n": 4096, "lo": 16, "hi": 64, "batch": 6},
        # a global layer of ModernBERT-base over a batch of documents of ordinary lengths
        {"name": "docs_global", **mha64, "dist": "lognormal", "n": 64, "median": 400, "lo": 32, "hi": 2048, "batch": 2},
        # the same documents in a local (+-64) layer, two layers of three
        {"name": "docs_band", **mha64, "window": HALF_WINDOW, "dist": "lognormal", "n": 64, "median": 400, "lo": 32,
         "hi": 2048, "batch": 2},
        # a contrastive batch: 512 queries beside 64 documents in one call
        {"name": "queries_and_docs", **mha64, "dist": "mixed", "n": 64, "median": 700, "lo": 256, "hi": 8192,
         "queries": 512, "query_lo": 8, "query_hi": 48, "batch": 3},
        # long documents at ModernBERT-large's head count: the largest attention call
        {"name": "long_global", **mha64, "hq": 16, "hkv": 16, "dist": "uniform", "n": 16, "lo": 8192, "hi": 8192,
         "batch": 0},
        # gated grouped-query layer of a hybrid decoder-style encoder: head_dim 256, causal
        {"name": "gated_gqa_256", "op": "attention", "hq": 8, "hkv": 2, "d": 256, "window": -1, "causal": True,
         "gate": True, "dist": "uniform", "n": 256, "lo": 16, "hi": 512, "batch": 5},
        # grouped-query causal prefill at head_dim 128, documents of ordinary lengths
        {"name": "causal_gqa_128", "op": "attention", "hq": 32, "hkv": 8, "d": 128, "window": -1, "causal": True,
         "gate": False, "dist": "lognormal", "n": 32, "median": 700, "lo": 64, "hi": 4096, "batch": 8},
        # requests that continue a cached prefix (decode steps and short tails) at head_dim 128
        {"name": "prefixed_gqa_128", "op": "prefixed", "hq": 32, "hkv": 8, "d": 128, "causal": True,
         "dist": "uniform", "n": 16, "lo": 512, "hi": 8192, "tail_lo": 1, "tail_hi": 32, "batch": 9},
        # one local ModernBERT-base layer over the documents: norms, products, RoPE, band, MLP
        {"name": "layer_docs", "op": "layer", **BASE, "global": False, "dist": "lognormal", "n": 64, "median": 400,
         "lo": 32, "hi": 2048, "batch": 2},
        # the whole encoder on a handful of online queries: launch-bound
        {"name": "forward_queries", "op": "forward", **BASE, "layers": 22, "dist": "uniform", "n": 8, "lo": 4, "hi": 32,
         "batch": 4},
        # the whole encoder on the batch of documents
        {"name": "forward_docs", "op": "forward", **BASE, "layers": 22, "dist": "lognormal", "n": 64, "median": 400,
         "lo": 32, "hi": 2048, "batch": 2},
    ]


def _log(rng, lo: float, hi: float) -> int:
    return max(int(lo), min(int(hi), round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    """One more case of the listed ones' ranges (sizes over their logarithm)."""
    batch = rng.randrange(1 << 30)
    heads = rng.choice((12, 16))
    mha64 = {"op": "attention", "hq": heads, "hkv": heads, "d": 64, "causal": False, "gate": False}
    docs = {"dist": "lognormal", "n": _log(rng, 4, 96), "median": _log(rng, 150, 1500), "lo": 32, "hi": 2048,
            "batch": batch}
    kind = rng.randrange(9)
    if kind == 0:  # short queries, one call
        return {**mha64, "window": rng.choice((-1, HALF_WINDOW)), "dist": "uniform", "n": _log(rng, 1, 2048),
                "lo": rng.randint(1, 16), "hi": rng.randint(17, 128), "batch": batch}
    if kind == 1:  # RoPE and attention: queries (fused) or documents (two kernels)
        short = {"dist": "uniform", "n": _log(rng, 8, 4096), "lo": rng.randint(1, 16), "hi": rng.randint(17, 128),
                 "batch": batch}
        return {"op": "rope_attention", "hq": 12, "d": 64, "window": rng.choice((-1, HALF_WINDOW)),
                **(short if rng.random() < 0.7 else docs)}
    if kind == 2:  # documents, global or local layer
        return {**mha64, "window": rng.choice((-1, HALF_WINDOW)), **docs}
    if kind == 3:  # queries and documents in one call
        return {**mha64, "window": -1, **docs, "dist": "mixed", "lo": 256, "hi": 8192, "n": _log(rng, 4, 48),
                "queries": _log(rng, 16, 1024), "query_lo": 4, "query_hi": rng.randint(24, 64)}
    if kind == 4:  # long documents
        return {**mha64, "window": rng.choice((-1, HALF_WINDOW)), "dist": "uniform", "n": _log(rng, 1, 12),
                "lo": 2049, "hi": _log(rng, 3000, 8192), "batch": batch}
    if kind == 5:  # gated head_dim 256
        return {"op": "attention", "hq": 8, "hkv": 2, "d": 256, "window": -1, "causal": True,
                "gate": rng.random() < 0.75, "dist": "uniform", "n": _log(rng, 8, 256), "lo": rng.randint(1, 64),
                "hi": _log(rng, 128, 1024), "batch": batch}
    if kind == 6:  # grouped-query head_dim 128
        hq, hkv = rng.choice(((32, 8), (16, 8), (16, 16)))
        return {"op": "attention", "hq": hq, "hkv": hkv, "d": 128, "window": -1, "causal": rng.random() < 0.75,
                "gate": False, "dist": "lognormal", "n": _log(rng, 4, 64), "median": _log(rng, 128, 1000), "lo": 33,
                "hi": 4096, "batch": batch}
    if kind == 7:  # continuing a prefix
        hq, hkv, d = rng.choice(((32, 8, 128), (16, 8, 128), (8, 2, 256), (12, 12, 64)))
        return {"op": "prefixed", "hq": hq, "hkv": hkv, "d": d, "causal": True, "dist": "uniform",
                "n": _log(rng, 1, 64), "lo": rng.randint(128, 600), "hi": _log(rng, 1000, 8192), "tail_lo": 1,
                "tail_hi": _log(rng, 1, 128), "batch": batch}
    # one layer
    shape = rng.choice((BASE, LARGE))
    queries = {"dist": "uniform", "n": _log(rng, 2, 512), "lo": 4, "hi": rng.randint(16, 128), "batch": batch}
    return {"op": "layer", **shape, "global": rng.random() < 0.4, **(queries if rng.random() < 0.4 else docs)}


# ----------------------------------------------------------------------------- sizes


def _lengths(case: dict) -> list[int]:
    """Segment lengths (key lengths of a ``prefixed`` case)."""
    rng = workloads.SplitMix64(case["batch"])
    if case["dist"] == "uniform":
        return [rng.randint(case["lo"], case["hi"]) for _ in range(case["n"])]
    first = []
    if case["dist"] == "mixed":
        first = [rng.randint(case["query_lo"], case["query_hi"]) for _ in range(case["queries"])]
    return first + [rng.lognormal_length(case["median"], 0.8, case["lo"], case["hi"]) for _ in range(case["n"])]


def _tails(case: dict) -> list[int]:
    rng = workloads.SplitMix64(case["batch"] + 1)
    return [rng.randint(case["tail_lo"], case["tail_hi"]) for _ in range(case["n"])]


def _window(case: dict) -> tuple[int, int]:
    w = case.get("window", -1)
    if case["op"] == "layer":
        w = -1 if case["global"] else HALF_WINDOW
    return (w, w)


def _pairs(lengths, window, causal) -> int:
    """Allowed (query, key) pairs: ``|i - j| <= window`` and, causal, ``j <= i``."""
    total = 0
    for n in lengths:
        w = n - 1 if window[0] < 0 else min(window[0], n - 1)
        below = n * w - w * (w + 1) // 2
        total += n + below * (1 if causal else 2)
    return total


def _dense(case: dict, tokens: int) -> tuple[int, int]:
    """(flops, weight elements) of one encoder layer's four products."""
    weights = case["hidden"] * (4 * case["hidden"] + 3 * case["mlp"])
    return 2 * tokens * weights, weights


def work(case: dict) -> dict:
    lengths = _lengths(case)
    tokens, op = sum(lengths), case["op"]
    if op == "prefixed":
        tails = _tails(case)
        pairs = sum(t * k - t * (t - 1) // 2 for t, k in zip(tails, lengths))
        return {"flops": 4 * case["d"] * case["hq"] * pairs,
                "bytes": 4 * case["d"] * (case["hq"] * sum(tails) + case["hkv"] * tokens)}
    if op == "attention":
        rows = (2 + bool(case["gate"])) * case["hq"] + 2 * case["hkv"]
        return {"flops": 4 * case["d"] * case["hq"] * _pairs(lengths, _window(case), case["causal"]),
                "bytes": 2 * tokens * case["d"] * rows}
    if op == "rope_attention":  # the projection and two table rows in, the context out
        return {"flops": 4 * case["d"] * case["hq"] * _pairs(lengths, _window(case), False),
                "bytes": 2 * tokens * case["d"] * (4 * case["hq"] + 2)}
    flops, weights = _dense(case, tokens)
    if op == "layer":
        flops += 4 * case["hidden"] * _pairs(lengths, _window(case), False)
        return {"flops": flops, "bytes": 2 * (4 * tokens * case["hidden"] + weights)}
    every, local = (_pairs(lengths, (w, w), False) for w in (-1, HALF_WINDOW))
    n_global = sum(1 for i in range(case["layers"]) if i % 3 == 0)
    flops = case["layers"] * flops + 4 * case["hidden"] * (n_global * every + (case["layers"] - n_global) * local)
    return {"flops": flops, "bytes": 2 * (2 * tokens * case["hidden"] + case["layers"] * weights)}


def tolerance(case: dict) -> dict:
    # bf16 outputs of fp32 sums over bf16 probabilities; a layer and the whole encoder round to
    # bf16 after every operation, and the encoder carries that through 22 layers
    return {"attention": {"rel": 0.01, "max": 0.1}, "prefixed": {"rel": 0.01, "max": 0.1},
            "rope_attention": {"rel": 0.012, "max": 0.1}, "layer": {"rel": 0.02, "max": 0.15},
            "forward": {"rel": 0.03, "max": 0.5}}[case["op"]]


# ----------------------------------------------------------------------------- inputs


def _cu(lengths) -> torch.Tensor:
    bounds = [0]
    for n in lengths:
        bounds.append(bounds[-1] + n)
    return torch.tensor(bounds, dtype=torch.int32, device="cuda")


def _positions(lengths) -> torch.Tensor:
    return torch.cat([torch.arange(n) for n in lengths]).cuda()


def _randn(gen, *shape, std: float = 1.0) -> torch.Tensor:
    return torch.empty(*shape, dtype=torch.bfloat16, device="cuda").normal_(0.0, std, generator=gen)


class _Norm(nn.Module):
    def __init__(self, gen, hidden):
        super().__init__()
        self.weight = nn.Parameter(1 + _randn(gen, hidden, std=0.1), requires_grad=False)
        self.eps = 1e-5


class _Weight(nn.Module):
    def __init__(self, gen, *shape):
        super().__init__()
        self.weight = nn.Parameter(_randn(gen, *shape, std=0.02), requires_grad=False)


class _Embedding(_Weight):
    def forward(self, ids):
        return nn.functional.embedding(ids, self.weight)


def _layer(gen, case, first: bool) -> nn.Module:
    """A ModernBERT layer's modules (the first layer has no attention norm)."""
    hidden, mlp = case["hidden"], case["mlp"]
    layer = nn.Module()
    layer.attn_norm = nn.Identity() if first else _Norm(gen, hidden)
    layer.attn, layer.mlp = nn.Module(), nn.Module()
    layer.attn.Wqkv, layer.attn.Wo = _Weight(gen, 3 * hidden, hidden), _Weight(gen, hidden, hidden)
    layer.mlp_norm = _Norm(gen, hidden)
    layer.mlp.Wi, layer.mlp.Wo = _Weight(gen, 2 * mlp, hidden), _Weight(gen, hidden, mlp)
    return layer


def _encoder(gen, case) -> nn.Module:
    model = nn.Module()
    model.embeddings = nn.Module()
    model.embeddings.tok_embeddings = _Embedding(gen, VOCAB, case["hidden"])
    model.embeddings.norm = _Norm(gen, case["hidden"])
    model.layers = nn.ModuleList(_layer(gen, case, i == 0) for i in range(case["layers"]))
    model.final_norm = _Norm(gen, case["hidden"])
    return model


def _params(case: dict) -> ModernBertParams:
    return ModernBertParams(hidden_size=case["hidden"], num_attention_heads=case["hq"],
                            num_hidden_layers=case.get("layers", 1), norm_eps=1e-5, global_rope_theta=THETA[True],
                            local_rope_theta=THETA[False], local_attention=2 * HALF_WINDOW,
                            global_attn_every_n_layers=3)


def prepare(case: dict, seed: int) -> dict:
    gen = torch.Generator(device="cuda").manual_seed(seed)
    lengths = _lengths(case)
    tokens, op = sum(lengths), case["op"]
    state = {"case": case, "cu": _cu(lengths), "max": max(lengths), "min": min(lengths)}
    if op in ("attention", "prefixed"):
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        if op == "prefixed":
            tails = [min(t, k) for t, k in zip(_tails(case), lengths)]
            state.update(cu_k=state["cu"], max_k=state["max"], cu=_cu(tails), max=max(tails),
                         q=_randn(gen, sum(tails), hq, d), k=_randn(gen, tokens, hkv, d), v=_randn(gen, tokens, hkv, d))
        elif hq == hkv and d == 64:
            qkv = _randn(gen, tokens, 3, hq, d)
            state.update(q=qkv[:, 0].contiguous(), k=qkv[:, 1].contiguous(), v=qkv[:, 2])
        else:
            state.update(q=_randn(gen, tokens, hq, d), k=_randn(gen, tokens, hkv, d), v=_randn(gen, tokens, hkv, d))
        state["gate"] = _randn(gen, tokens, hq, d) if case.get("gate") else None
        return state
    if op == "forward":
        ids = torch.empty(tokens, dtype=torch.long, device="cuda").random_(VOCAB, generator=gen)
        return {**state, "model": _encoder(gen, case), "params": _params(case), "ids": ids,
                "positions": _positions(lengths)}
    d = 64
    is_global = case["global"] if op == "layer" else case["window"] < 0
    tables = ops.rope_tables(state["max"], d, THETA[is_global], torch.device("cuda"), torch.bfloat16)
    positions = _positions(lengths)
    state["cos"], state["sin"] = (t[0].index_select(0, positions)[None] for t in tables)
    if op == "rope_attention":
        return {**state, "qkv": _randn(gen, 1, tokens, 3 * case["hq"] * d)}
    return {**state, "layer": _layer(gen, case, False), "params": _params(case),
            "x": _randn(gen, 1, tokens, case["hidden"]), "residual": _randn(gen, 1, tokens, case["hidden"], std=0.5),
            "execution": pe.pieces.default_execution()}


def run(state: dict):
    case, cu, longest = state["case"], state["cu"], state["max"]
    with torch.no_grad():
        if case["op"] == "attention":
            return pe.varlen_attention(state["q"], state["k"], state["v"], cu, longest, window=_window(case),
                                       causal=case["causal"], gate=state["gate"], min_seqlen=state["min"])
        if case["op"] == "prefixed":
            return pe.varlen_attention(state["q"], state["k"], state["v"], cu, longest, causal=case["causal"],
                                       cu_seqlens_k=state["cu_k"], max_seqlen_k=state["max_k"])
        if case["op"] == "rope_attention":
            return ops.flash_attention_qkv_bshd(state["qkv"], case["hq"], case["d"], cos=state["cos"],
                                                sin=state["sin"], window=_window(case), scaling=case["d"] ** -0.5,
                                                cu_seqlens=cu, max_seqlen=longest)
        if case["op"] == "layer":
            kind = forward.LayerKind(state["cos"], state["sin"], None, _window(case))
            return forward.encoder_layer(state["x"], state["residual"], state["layer"], state["params"], kind, "hip",
                                         state["execution"], cu_seqlens=cu, max_seqlen=longest)
        return pe.packed_forward(state["model"], state["params"], state["ids"], cu, longest, state["positions"],
                                 min_seqlen=state["min"])


# ----------------------------------------------------------------------------- 64-bit results


def _attend(q, k, v, window, causal: bool, scale: float):
    """One segment in float64: q ``[Lq, Hq, D]``, k and v ``[Lk, Hkv, D]``, queries end-aligned."""
    group = q.shape[1] // k.shape[1]
    lq, lk = q.shape[0], k.shape[0]
    mask = None
    if causal or window[0] >= 0:
        ahead = torch.arange(lk, device=q.device)[None] - (torch.arange(lq, device=q.device) + lk - lq)[:, None]
        mask = (ahead > 0) if causal else (ahead.abs() > window[0])
    out = torch.empty_like(q)
    for h in range(0, k.shape[1], max(1, 4096 * 4096 // (lq * lk))):
        part = slice(h, min(k.shape[1], h + max(1, 4096 * 4096 // (lq * lk))))
        qh = q.transpose(0, 1)[part.start * group:part.stop * group].contiguous()
        kh, vh = (t.transpose(0, 1)[part].repeat_interleave(group, dim=0).contiguous() for t in (k, v))
        s = torch.matmul(qh, kh.transpose(1, 2).contiguous()).mul_(scale)
        if mask is not None:
            s.masked_fill_(mask, float("-inf"))
        out[:, part.start * group:part.stop * group] = torch.matmul(torch.softmax(s, -1), vh).transpose(0, 1)
    return out


def _packed(q, k, v, lengths, lengths_k, window, causal):
    out = torch.empty_like(q)
    at = at_k = 0
    for n, m in zip(lengths, lengths_k):
        part = slice(at_k, at_k + m)
        out[at:at + n] = _attend(q[at:at + n], k[part], v[part], window, causal, q.shape[-1] ** -0.5)
        at, at_k = at + n, at_k + m
    return out


def _rotated(x, cos, sin):
    half = x.shape[-1] // 2
    swapped = torch.cat((-x[..., half:], x[..., :half]), -1)
    return x * cos[:, None] + swapped * sin[:, None]


def _from_qkv(qkv, heads, cos, sin, lengths, window):
    q, k, v = qkv.view(qkv.shape[0], 3, heads, -1).unbind(1)
    out = _packed(_rotated(q, cos, sin), _rotated(k, cos, sin), v, lengths, lengths, window, False)
    return out.reshape(qkv.shape[0], -1)


def _normed(x, norm):
    return nn.functional.layer_norm(x, (x.shape[-1],), norm.weight.double(), None, norm.eps)


def _exact_layer(x, residual, layer, heads, cos, sin, lengths, window):
    if residual is not None:
        x = x + residual
    normed = x if isinstance(layer.attn_norm, nn.Identity) else _normed(x, layer.attn_norm)
    ctx = _from_qkv(normed @ layer.attn.Wqkv.weight.double().t(), heads, cos, sin, lengths, window)
    x = x + ctx @ layer.attn.Wo.weight.double().t()
    inp, gate = (_normed(x, layer.mlp_norm) @ layer.mlp.Wi.weight.double().t()).chunk(2, -1)
    return x, (nn.functional.gelu(inp) * gate) @ layer.mlp.Wo.weight.double().t()


def _exact_tables(theta: float, d: int, positions):
    freq = theta ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
    angles = positions.double()[:, None] * freq[None]
    angles = torch.cat((angles, angles), -1)
    return angles.cos(), angles.sin()


def exact(case: dict, seed: int):
    state = prepare(case, seed)
    lengths = _lengths(case)
    with torch.no_grad():
        if case["op"] in ("attention", "prefixed"):
            rows = lengths
            if case["op"] == "prefixed":
                rows = [min(t, k) for t, k in zip(_tails(case), lengths)]
            out = _packed(state["q"].double(), state["k"].double(), state["v"].double(), rows, lengths, _window(case),
                          case["causal"])
            return out if state["gate"] is None else out * torch.sigmoid(state["gate"].double())
        if case["op"] == "rope_attention":
            return _from_qkv(state["qkv"][0].double(), case["hq"], state["cos"][0].double(), state["sin"][0].double(),
                             lengths, _window(case))[None]
        if case["op"] == "layer":
            out = _exact_layer(state["x"][0].double(), state["residual"][0].double(), state["layer"], case["hq"],
                               state["cos"][0].double(), state["sin"][0].double(), lengths, _window(case))
            return tuple(t[None] for t in out)
        model = state["model"]
        tables = {g: _exact_tables(THETA[g], 64, state["positions"]) for g in (True, False)}
        x = _normed(model.embeddings.tok_embeddings.weight[state["ids"]].double(), model.embeddings.norm)
        residual = None
        for i, layer in enumerate(model.layers):
            is_global = i % 3 == 0
            w = -1 if is_global else HALF_WINDOW
            x, residual = _exact_layer(x, residual, layer, case["hq"], *tables[is_global], lengths, (w, w))
        return _normed(x + residual, model.final_norm)
