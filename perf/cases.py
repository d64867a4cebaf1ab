"""The work a program has this library do, as measurable cases.

A case is a dict of plain values. ``listed()`` gives the fixed ones, ``draw``
one more from the ranges they stand for, ``prepare`` what a program holds
before the call, ``run`` one pass through the public entry points, ``work``
the bytes and operations a pass cannot do without, ``exact`` its results in 64
bits and ``tolerance`` how far a correct implementation may be from them.

Ranges (``draw``):

* norm        RMSNorm, plain and residual: 1-16384 rows of 256-16384 elements,
              any width, float16 / bfloat16 / float32, weights in the input's
              type or float32, rows dense or cut out of wider ones;
* head_norm   RMSNorm over each attention head: up to 262144 rows of 32-256;
* shard_norm  one tensor-parallel rank's part of a residual RMSNorm;
* rope        query and key rotated together: both pairings, head sizes of
              32-256, grouped keys, separate or cut out of a fused projection;
* rope_cache  the same with the key/value cache append, one token or many;
* swiglu      1-16384 rows of 256-16384, dense or the halves of one projection;
* prefill     a whole decoder's prompt pass, 16-512 tokens.
"""

from __future__ import annotations

import math

import torch

import ako_amd as ako
from ako_amd.models.decoder import ModelConfig, build_lm
from ako_amd.ops.rmsnorm_tp import rmsnorm_shard_apply_hip, rmsnorm_shard_partial_hip
from ako_amd.ops.rope import rope_qk_cache

DEVICE = "cuda"
EPS = 1e-6
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
#: Elements per tensor of the largest case; no drawn case has more.
MAX_ELEMENTS = 16384 * 16384
#: The decoder's per-operation override: the kernels themselves, not the
#: selector's timing of them, are what a case measures.
OVERRIDE = {"rmsnorm": "rmsnorm_hip", "rmsnorm_residual": "rmsnorm_residual_hip", "swiglu": "swiglu_hip"}


# --------------------------------------------------------------------- cases --
def norm_case(rows, hidden, dtype, *, residual, weight="same", pad=0):
    return {"kind": "norm", "rows": rows, "hidden": hidden, "dtype": dtype, "residual": residual,
            "weight": weight, "pad": pad}


def head_norm_case(batch, seq, heads, head_dim, dtype):
    return {"kind": "head_norm", "batch": batch, "seq": seq, "heads": heads, "head_dim": head_dim, "dtype": dtype}


def shard_norm_case(rows, hidden, ranks, dtype):
    return {"kind": "shard_norm", "rows": rows, "hidden": hidden, "ranks": ranks, "dtype": dtype}


def rope_case(batch, seq, heads, kv_heads, head_dim, dtype, *, style, tables="same", fused=False):
    return {"kind": "rope", "batch": batch, "seq": seq, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim,
            "dtype": dtype, "style": style, "tables": tables, "fused": fused}


def rope_cache_case(batch, seq, heads, kv_heads, head_dim, cache_len, pos, dtype, *, style="neox"):
    return {"kind": "rope_cache", "batch": batch, "seq": seq, "heads": heads, "kv_heads": kv_heads,
            "head_dim": head_dim, "cache_len": cache_len, "pos": pos, "dtype": dtype, "style": style}


def swiglu_case(rows, width, dtype, *, fused=False):
    return {"kind": "swiglu", "rows": rows, "width": width, "dtype": dtype, "fused": fused}


def prefill_case(tokens, kv_heads):
    return {"kind": "prefill", "tokens": tokens, "kv_heads": kv_heads}


def listed() -> list[dict]:
    return [
        # One token of a decode step: the smallest call, all latency and launch.
        {"name": "norm_decode", **norm_case(1, 4096, "float16", residual=True)},
        # The norm before a block over an ordinary prompt batch, at the width of
        # a 13B-class model (not a power of two).
        {"name": "norm_prompt", **norm_case(4096, 5120, "bfloat16", residual=True)},
        # Long-context prefill at the widest hidden size: the largest call.
        {"name": "norm_widest", **norm_case(16384, 16384, "bfloat16", residual=True)},
        # Rows of no round size, as pruned or unpadded models have them; every
        # second row starts off a 16-byte boundary.
        {"name": "norm_ragged", **norm_case(2049, 4099, "float16", residual=False)},
        # Query norm per attention head: many short rows.
        {"name": "norm_heads", **head_norm_case(4, 2048, 32, 128, "bfloat16")},
        # One of 8 tensor-parallel ranks: its slice's sums, then its slice's output.
        {"name": "norm_shard", **shard_norm_case(16384, 16384, 8, "bfloat16")},
        # Prompt batch with grouped keys, q and k cut out of a fused projection.
        {"name": "rope_prompt", **rope_case(4, 2048, 32, 8, 128, "float16", style="neox", fused=True)},
        # Interleaved pairing in full precision, an odd length, a head size that
        # is not a power of two.
        {"name": "rope_pairs", **rope_case(3, 1025, 32, 32, 80, "float32", style="interleaved")},
        # A serving batch's decode step: rotate and append one token each.
        {"name": "rope_append", **rope_cache_case(64, 1, 32, 8, 128, 640, 512, "float16")},
        # The MLP's activation over an ordinary prompt batch, two projections.
        {"name": "swiglu_prompt", **swiglu_case(4096, 14336, "bfloat16")},
        # The same from one fused gate/up projection's two halves, odd token count.
        {"name": "swiglu_halves", **swiglu_case(3001, 5632, "float16", fused=True)},
        # A four-layer decoder's prompt pass, through every operation.
        {"name": "decoder_prefill", **prefill_case(512, 32)},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _width(rng, lo: int, hi: int) -> int:
    """A row width: mostly the multiples of 128 that models have, some of 8, some of nothing."""
    w = _log_int(rng, lo, hi)
    step = rng.choice([128, 128, 8, 1])
    return min(hi, max(lo, round(w / step) * step))


def draw(rng) -> dict:
    kind = rng.choice(["norm", "norm", "norm", "head_norm", "shard_norm", "rope", "rope", "rope_cache", "swiglu",
                       "swiglu", "prefill"])
    dtype = rng.choice(["float16", "bfloat16", "bfloat16", "float32"])
    half = rng.choice(["float16", "bfloat16"])
    if kind == "norm":
        hidden = _width(rng, 256, 16384)
        rows = _log_int(rng, 1, 16384)
        if dtype == "float32":
            rows = min(rows, MAX_ELEMENTS // 2 // hidden)
        return norm_case(rows, hidden, dtype, residual=rng.random() < 0.5,
                         weight=rng.choice(["same", "same", "float32"]), pad=rng.choice([0, 0, 0, 64]))
    if kind == "head_norm":
        heads = rng.choice([8, 16, 32, 40])
        tokens = _log_int(rng, 1, 8192)
        batch = rng.choice([1, 2, 3, 4])
        return head_norm_case(batch, max(1, tokens // batch), heads, rng.choice([32, 64, 80, 96, 128, 192, 256]), dtype)
    if kind == "shard_norm":
        ranks = rng.choice([2, 4, 8])
        return shard_norm_case(_log_int(rng, 1, 16384), ranks * _width(rng, 256, 16384 // ranks), ranks, half)
    if kind in ("rope", "rope_cache"):
        heads = rng.choice([8, 16, 32, 40])
        kv_heads = rng.choice([heads, heads // 4, heads // 8])
        head_dim = rng.choice([32, 64, 64, 72, 80, 96, 128, 128, 192, 256])
        style = rng.choice(["neox", "neox", "interleaved"])
        batch = rng.choice([1, 2, 3, 4])
        if kind == "rope":
            seq = max(1, _log_int(rng, 1, 8192) // batch)
            return rope_case(batch, seq, heads, kv_heads, head_dim, dtype, style=style,
                             tables=rng.choice(["same", "float32"]), fused=rng.random() < 0.5)
        cache_len = rng.choice([640, 2048])
        if rng.random() < 0.6:
            batch, seq = _log_int(rng, 1, 64), 1
        else:
            seq = _log_int(rng, 2, cache_len // 2)
        batch = max(1, min(batch, (1 << 25) // (kv_heads * cache_len * head_dim)))
        return rope_cache_case(batch, seq, heads, kv_heads, head_dim, cache_len, rng.randrange(cache_len - seq + 1),
                               half, style=style)
    if kind == "swiglu":
        return swiglu_case(_log_int(rng, 1, 16384), _width(rng, 256, 16384), half if rng.random() < 0.75 else dtype,
                           fused=rng.random() < 0.4)
    return prefill_case(_log_int(rng, 16, 512), rng.choice([8, 32]))


# ------------------------------------------------------------------- prepare --
class Inputs:
    """Seeded tensors; each call draws the next ones."""

    def __init__(self, seed: int):
        self.gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def activations(self, shape, dtype, scale=1.0):
        out = torch.empty(shape, dtype=DTYPES[dtype], device=DEVICE)
        out.normal_(0.0, scale, generator=self.gen)
        return out

    def norm_weight(self, width, dtype):
        w = torch.empty(width, dtype=torch.float32, device=DEVICE)
        return w.normal_(1.0, 0.1, generator=self.gen).to(DTYPES[dtype])


def _rope_tables(positions: int, case: dict):
    dtype = case["dtype"] if case.get("tables", "same") == "same" else case["tables"]
    cos, sin = ako.build_rope_tables(positions, case["head_dim"], device=DEVICE, dtype=torch.float32)
    return cos.to(DTYPES[dtype]), sin.to(DTYPES[dtype])


def _qkv(inputs: Inputs, case: dict, fused: bool, dtype: str):
    """q, k and v of (batch, seq, heads, head_dim): one projection's columns, or three tensors."""
    b, s, d = case["batch"], case["seq"], case["head_dim"]
    counts = (case["heads"], case["kv_heads"], case["kv_heads"])
    if not fused:
        return [inputs.activations((b, s, n, d), dtype) for n in counts]
    whole = inputs.activations((b, s, sum(counts) * d), dtype)
    return [part.view(b, s, n, d) for part, n in zip(whole.split([n * d for n in counts], -1), counts)]


def _model_config(case: dict) -> ModelConfig:
    return ModelConfig(hidden_dim=4096, n_layers=4, n_heads=32, n_kv_heads=case["kv_heads"], intermediate_dim=11008,
                       max_seq_len=1024, rope_base=10000.0, eps=EPS, vocab_size=32000)


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    inputs = Inputs(seed)
    state = {"case": case}
    if kind == "norm":
        rows, hidden, pad = case["rows"], case["hidden"], case["pad"]
        dtype = case["dtype"]
        state["x"] = inputs.activations((rows, hidden + pad), dtype)[:, :hidden]
        if case["residual"]:  # the residual stream grows through the layers
            state["residual"] = inputs.activations((rows, hidden + pad), dtype, 2.0)[:, :hidden]
        state["weight"] = inputs.norm_weight(hidden, dtype if case["weight"] == "same" else case["weight"])
    elif kind == "head_norm":
        shape = (case["batch"], case["seq"], case["heads"], case["head_dim"])
        state["x"] = inputs.activations(shape, case["dtype"])
        state["weight"] = inputs.norm_weight(case["head_dim"], case["dtype"])
    elif kind == "shard_norm":
        rows, width, dtype = case["rows"], case["hidden"] // case["ranks"], case["dtype"]
        state["x"] = inputs.activations((rows, width), dtype)
        state["residual"] = inputs.activations((rows, width), dtype, 2.0)
        state["weight"] = inputs.norm_weight(width, dtype)
        # What the other ranks' slices add to each row's sum of squares.
        others = torch.empty(rows, dtype=torch.float32, device=DEVICE).uniform_(4.9, 5.1, generator=inputs.gen)
        state["others"] = others * (case["hidden"] - width)
    elif kind == "rope":
        state["q"], state["k"], _ = _qkv(inputs, case, case["fused"], case["dtype"])
        state["cos"], state["sin"] = _rope_tables(case["seq"], case)
    elif kind == "rope_cache":
        state["q"], state["k"], state["v"] = _qkv(inputs, case, True, case["dtype"])
        state["cos"], state["sin"] = _rope_tables(case["cache_len"], {**case, "tables": "float32"})
        shape = (case["batch"], case["kv_heads"], case["cache_len"], case["head_dim"])
        state["k_cache"] = inputs.activations(shape, case["dtype"])
        state["v_cache"] = inputs.activations(shape, case["dtype"])
        state["pos"] = torch.full((1,), case["pos"], dtype=torch.long, device=DEVICE)
    elif kind == "swiglu":
        rows, width, dtype = case["rows"], case["width"], case["dtype"]
        if case["fused"]:
            both = inputs.activations((rows, 2 * width), dtype, 2.0)
            state["gate"], state["up"] = both[:, :width], both[:, width:]
        else:
            state["gate"] = inputs.activations((rows, width), dtype, 2.0)
            state["up"] = inputs.activations((rows, width), dtype, 2.0)
    else:
        state["model"] = build_lm(_model_config(case), device=DEVICE, dtype=torch.float16, seed=seed,
                                  kernel_override=OVERRIDE)
        state["ids"] = torch.randint(0, 32000, (1, case["tokens"]), generator=inputs.gen, device=DEVICE)
    return state


# ----------------------------------------------------------------------- run --
@torch.no_grad()
def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "norm" and case["residual"]:
        return ako.rmsnorm_residual(state["x"], state["residual"], state["weight"], EPS,
                                    kernel="rmsnorm_residual_hip")
    if kind in ("norm", "head_norm"):
        return ako.rmsnorm(state["x"], state["weight"], EPS, kernel="rmsnorm_hip")
    if kind == "shard_norm":
        total_stream, sums = rmsnorm_shard_partial_hip(state["x"], state["residual"])
        sums.add_(state["others"])  # where a rank all-reduces
        y = rmsnorm_shard_apply_hip(total_stream, state["weight"], sums, case["hidden"], EPS)
        return y, total_stream, sums
    if kind == "rope":
        return ako.rope_qk(state["q"], state["k"], state["cos"], state["sin"], case["style"], kernel="rope_qk_hip")
    if kind == "rope_cache":
        q = rope_qk_cache(state["q"], state["k"], state["v"], state["cos"], state["sin"], state["pos"],
                          state["k_cache"], state["v_cache"], case["style"])
        return q, state["k_cache"], state["v_cache"]
    if kind == "swiglu":
        return ako.swiglu(state["gate"], state["up"], kernel="swiglu_hip")
    model, ids = state["model"], state["ids"]
    cache = model.stack.new_kv_cache(case["tokens"] + 128)
    logits = model.logits_last(ids, cache)
    filled = [(k[:, : cache.length], v[:, : cache.length]) for k, v in cache.entries]
    return {"logits": logits, "keys": [k for k, _ in filled], "values": [v for _, v in filled]}


# ---------------------------------------------------------------------- work --
def _size(dtype: str) -> int:
    return DTYPES[dtype].itemsize


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "norm":
        n, e = case["rows"] * case["hidden"], _size(case["dtype"])
        weight = case["hidden"] * (e if case["weight"] == "same" else 4)
        return {"bytes": n * e * (4 if case["residual"] else 2) + weight, "flops": n * (5 if case["residual"] else 4)}
    if kind == "head_norm":
        n, e = case["batch"] * case["seq"] * case["heads"] * case["head_dim"], _size(case["dtype"])
        return {"bytes": 2 * n * e + case["head_dim"] * e, "flops": 4 * n}
    if kind == "shard_norm":
        width, e = case["hidden"] // case["ranks"], _size(case["dtype"])
        n = case["rows"] * width
        # The sums leave for the other ranks between the halves, so the summed
        # stream is written by the first half and read again by the second.
        return {"bytes": 5 * n * e + width * e + 12 * case["rows"], "flops": 5 * n}
    if kind == "rope":
        per_token = (case["heads"] + case["kv_heads"]) * case["head_dim"]
        n, e = case["batch"] * case["seq"] * per_token, _size(case["dtype"])
        table = case["seq"] * case["head_dim"] * (e if case["tables"] == "same" else 4)
        return {"bytes": 2 * n * e + table, "flops": 3 * n}
    if kind == "rope_cache":
        tokens, d, e = case["batch"] * case["seq"], case["head_dim"], _size(case["dtype"])
        n = tokens * (case["heads"] + 2 * case["kv_heads"]) * d
        return {"bytes": 2 * n * e + case["seq"] * d * 4 + 8,
                "flops": 3 * tokens * (case["heads"] + case["kv_heads"]) * d}
    if kind == "swiglu":
        n, e = case["rows"] * case["width"], _size(case["dtype"])
        return {"bytes": 3 * n * e, "flops": 6 * n}
    cfg, t = _model_config(case), case["tokens"]
    kv = cfg.n_kv_heads * cfg.head_dim
    layer = cfg.hidden_dim * (2 * cfg.hidden_dim + 2 * kv + 3 * cfg.intermediate_dim)
    head = cfg.hidden_dim * cfg.vocab_size
    attention = 2 * cfg.hidden_dim * t * t  # two products over the causal half
    return {"bytes": 2 * (cfg.n_layers * (layer + 2 * t * kv) + head + t * cfg.hidden_dim + cfg.vocab_size),
            "flops": cfg.n_layers * (2 * t * layer + attention) + 2 * head}


# --------------------------------------------------------------------- exact --
F64 = torch.float64
#: Elements per 64-bit block of a row-wise result (bounds the memory it takes).
BLOCK = 1 << 27


def _by_rows(fn, *tensors):
    """fn over blocks of the tensors' rows, the results joined."""
    step = max(1, BLOCK // tensors[0].shape[-1])
    parts = [fn(*(t[i:i + step] for t in tensors)) for i in range(0, tensors[0].shape[0], step)]
    if isinstance(parts[0], tuple):
        return tuple(torch.cat(p) for p in zip(*parts))
    return torch.cat(parts)


def _norm64(x, weight, mean_square=None):
    x = x.to(F64)
    if mean_square is None:
        mean_square = x.square().mean(-1, keepdim=True)
    return x * torch.rsqrt(mean_square + EPS) * weight.to(F64)


def _rotate64(x, cos, sin, style):
    """x (batch, seq, heads, head_dim) by (seq, head_dim / 2) tables."""
    x, c, n = x.to(F64), cos.to(F64)[:, None, :], sin.to(F64)[:, None, :]
    if style == "neox":
        a, b = x.chunk(2, -1)
        return torch.cat([a * c - b * n, a * n + b * c], -1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * n, a * n + b * c], -1).flatten(-2)


def _prefill64(model, ids, case):
    """The decoder in 64 bits from the model's own weights, layer by layer."""
    cfg = _model_config(case)
    t, heads, kv_heads, d = case["tokens"], cfg.n_heads, cfg.n_kv_heads, cfg.head_dim
    half = d // 2
    inv_freq = 1.0 / (10000.0 ** (torch.arange(half, device=DEVICE, dtype=torch.float32) * 2.0 / d))
    angles = torch.outer(torch.arange(t, device=DEVICE, dtype=torch.float32), inv_freq)
    cos, sin = angles.cos(), angles.sin()
    mask = torch.full((t, t), float("-inf"), dtype=F64, device=DEVICE).triu(1)
    h = model.embed.weight[ids[0]].to(F64)
    keys, values = [], []
    for layer in model.stack.layers:
        x = _norm64(h, layer.input_norm_weight)
        qkv = x @ layer.attention.qkv_proj.weight.to(F64).t()
        q, k, v = qkv.split([heads * d, kv_heads * d, kv_heads * d], -1)
        q = _rotate64(q.reshape(1, t, heads, d), cos, sin, "neox")[0]
        k = _rotate64(k.reshape(1, t, kv_heads, d), cos, sin, "neox")[0]
        v = v.reshape(t, kv_heads, d)
        keys.append(k[None])
        values.append(v[None])
        per_head = []
        for i in range(heads):
            j = i // (heads // kv_heads)
            scores = q[:, i].contiguous() @ k[:, j].t().contiguous() / math.sqrt(d) + mask
            per_head.append(torch.softmax(scores, -1) @ v[:, j].contiguous())
        h = h + torch.cat(per_head, -1) @ layer.attention.o_proj.weight.to(F64).t()
        x = _norm64(h, layer.post_attention_norm_weight)
        gate = x @ layer.mlp.gate_proj.weight.to(F64).t()
        up = x @ layer.mlp.up_proj.weight.to(F64).t()
        h = h + (gate * torch.sigmoid(gate) * up) @ layer.mlp.down_proj.weight.to(F64).t()
    x = _norm64(h, model.stack.final_norm_weight)
    return {"logits": x[-1:] @ model.lm_head.weight.to(F64).t(), "keys": keys, "values": values}


@torch.no_grad()
def exact(case: dict, seed: int):
    kind = case["kind"]
    state = prepare(case, seed)
    if kind in ("norm", "head_norm"):
        w = state["weight"]
        if kind == "head_norm" or not case["residual"]:
            return _by_rows(lambda x: _norm64(x, w), state["x"])

        def both(x, r):
            # The sum is rounded to the storage type before it is normalised:
            # that rounding is part of the operation.
            return _norm64(x + r, w), x.to(F64) + r.to(F64)

        return _by_rows(both, state["x"], state["residual"])
    if kind == "shard_norm":
        w, hidden = state["weight"], case["hidden"]

        def part(x, r, others):
            rounded = (x + r).to(F64)
            sums = rounded.square().sum(-1) + others.to(F64)
            return _norm64(rounded, w, sums.unsqueeze(-1) / hidden), x.to(F64) + r.to(F64), sums

        return _by_rows(part, state["x"], state["residual"], state["others"])
    if kind == "rope":
        cos, sin, style = state["cos"], state["sin"], case["style"]
        return _rotate64(state["q"], cos, sin, style), _rotate64(state["k"], cos, sin, style)
    if kind == "rope_cache":
        rows = slice(case["pos"], case["pos"] + case["seq"])
        cos, sin, style = state["cos"][rows], state["sin"][rows], case["style"]
        k_cache, v_cache = state["k_cache"].to(F64), state["v_cache"].to(F64)
        k_cache[:, :, rows] = _rotate64(state["k"], cos, sin, style).transpose(1, 2)
        v_cache[:, :, rows] = state["v"].to(F64).transpose(1, 2)
        return _rotate64(state["q"], cos, sin, style), k_cache, v_cache
    if kind == "swiglu":
        return _by_rows(lambda g, u: g.to(F64) * torch.sigmoid(g.to(F64)) * u.to(F64), state["gate"], state["up"])
    return _prefill64(state["model"], state["ids"], case)


# ----------------------------------------------------------------- tolerance --
def tolerance(case: dict) -> dict:
    """About four times the distance of one correct result from the exact one."""
    if case["kind"] == "prefill":  # four layers of 16-bit products and roundings
        return {"rel": 1.2e-2}
    return {"rel": {"float16": 1e-3, "bfloat16": 8e-3, "float32": 1e-6}[case["dtype"]]}
