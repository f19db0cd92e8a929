"""The work that a program using this library has it do, as cases to time and to check.

A case is a dict of plain values; "kind" says which public entry point it goes through:

* ``attend``   ``ops.paged_attention``: decode (rows = 1) or verify (rows = k+1) over a filled
               paged cache, all layers of the case in one call, one sequence or a ragged batch;
* ``step``     ``PagedKVCache.append_attend`` once per layer: the engine's decode or verify step,
               which writes the new tokens and attends over the context that includes them --
               eager, or recorded into a HIP graph and replayed (``graph``);
* ``prefill``  the same entry point with a chunk of prompt rows;
* ``quant``    ``ops.quant_append``: a prompt chunk quantized and written into every layer;
* ``fill``     ``PagedKVCache.prefill``: whole prompts of different lengths, packed;
* ``op``       ``ops.attention``: the contiguous (payload, scale) cache of the reference's op.

Head shapes are the Qwen2.5 ones the rest of the repository uses (12/2/128 and 14/2/64).
"""
import math
import random
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parents[1] / "specdec-context-scaling_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from specdec_amd.engine.paged_cache import PagedKVCache  # noqa: E402
from specdec_amd.kernels import ops  # noqa: E402

_TARGET = {"heads": 12, "kv": 2, "dim": 128}
_DRAFT = {"heads": 14, "kv": 2, "dim": 64}
_BLOCK = 16


def listed():
    return [
        # one layer of a short context: what one attention call costs when there is little to read
        {"name": "decode_1x2048", "kind": "attend", **_TARGET, "layers": 1, "batch": 1, "rows": 1, "lo": 2048, "hi": 2048},
        # single-token decode of the 28-layer target at 8K, one call for all layers
        {"name": "decode_28x8192", "kind": "attend", **_TARGET, "layers": 28, "batch": 1, "rows": 1, "lo": 8192, "hi": 8192},
        # the target's speculative verify: four drafted tokens and one more
        {"name": "verify_28x4096", "kind": "attend", **_TARGET, "layers": 28, "batch": 1, "rows": 5, "lo": 4096, "hi": 4096},
        # the draft model's decode, at a length that is no multiple of a page
        {"name": "draft_24x8191", "kind": "attend", **_DRAFT, "layers": 24, "batch": 1, "rows": 1, "lo": 8191, "hi": 8191},
        # one layer of a serving batch: 32 sequences of 2K to 32K tokens
        {"name": "batch32_ragged", "kind": "attend", **_TARGET, "layers": 1, "batch": 32, "rows": 1, "lo": 2048, "hi": 32768},
        # the engine's verify step, called layer by layer: append the five tokens and attend
        {"name": "step_target_verify", "kind": "step", **_TARGET, "layers": 28, "batch": 1, "rows": 5, "lo": 8192, "hi": 8192, "graph": False},
        # the engine's draft step, recorded once and replayed for every token
        {"name": "step_draft_graph", "kind": "step", **_DRAFT, "layers": 24, "batch": 1, "rows": 1, "lo": 8190, "hi": 8190, "graph": True},
        # the last 2048-token chunk of an 8K prompt, one layer of the target
        {"name": "prefill_target", "kind": "prefill", **_TARGET, "batch": 1, "rows": 2048, "lo": 8192, "hi": 8192},
        # the odd tail of a prompt on the draft model
        {"name": "prefill_draft_tail", "kind": "prefill", **_DRAFT, "batch": 1, "rows": 777, "lo": 5000, "hi": 5000},
        # a 2048-token chunk written into all 28 layers
        {"name": "quant_28x2048", "kind": "quant", **_TARGET, "layers": 28, "tokens": 2048, "with_k": True},
        # a batch of whole prompts of 100 to 4000 tokens, packed back to back, layer after layer
        {"name": "fill_ragged", "kind": "fill", **_TARGET, "layers": 28, "batch": 8, "lo": 100, "hi": 4000},
        # the reference's own op over its contiguous cache
        {"name": "op_verify", "kind": "op", **_TARGET, "batch": 1, "rows": 5, "lo": 4097, "hi": 4097},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over the logarithm, odd ones among them."""
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["attend", "attend", "attend", "step", "step", "prefill", "prefill", "quant", "fill", "op"])
        case = {"kind": kind, **rng.choice([_TARGET, _DRAFT])}
        if kind in ("attend", "step"):
            batch = rng.choice([1, 1, _log(rng, 2, 32)])
            lo = _log(rng, 64, 32768)
            hi = lo if batch == 1 else _log(rng, lo, 32768)
            case.update(layers=rng.choice([1, _log(rng, 2, 28), 24 if case["dim"] == 64 else 28]), batch=batch,
                        rows=rng.choice([1, 1, 5, rng.randint(2, 8)]), lo=lo, hi=hi)
            if batch > 1:
                case["lengths"] = rng.randrange(1 << 20)
            if kind == "step":
                case["graph"] = batch == 1 and rng.random() < 0.5
        elif kind == "prefill":
            batch = rng.choice([1, 1, 2])
            rows = _log(rng, 80, 2048)
            lo = _log(rng, rows, 16384)
            hi = lo if batch == 1 else _log(rng, lo, 16384)
            case.update(batch=batch, rows=rows, lo=lo, hi=hi)
            if batch > 1:
                case["lengths"] = rng.randrange(1 << 20)
        elif kind == "quant":
            case.update(layers=rng.choice([1, _log(rng, 2, 28)]), tokens=_log(rng, 16, 8192), with_k=rng.random() < 0.7)
        elif kind == "fill":
            lo = _log(rng, 20, 1000)
            case.update(layers=rng.choice([1, _log(rng, 2, 28)]), batch=_log(rng, 1, 48), lo=lo, hi=_log(rng, lo, 8192), lengths=rng.randrange(1 << 20))
        else:
            lo = _log(rng, 64, 16384)
            case.update(batch=rng.choice([1, 1, 2, 4]), rows=rng.choice([1, 5, rng.randint(2, 8)]), lo=lo, hi=lo)
        if _cost(case) <= most:
            return case


# ---------------------------------------------------------------------------- sizes
def _lengths(case):
    """Context length of every sequence, the new tokens among them; the first has the longest."""
    if case["lo"] == case["hi"]:
        return [case["lo"]] * case["batch"]
    rng = random.Random(case.get("lengths", 41))
    return [case["hi"]] + [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"] - 1)]


def _visible(t, s):
    """(query row, key) pairs of s rows over t keys under the offset-causal mask."""
    return s * (t - s) + s * (s + 1) // 2


def work(case):
    h, kv, d = case["heads"], case["kv"], case["dim"]
    page = kv * (2 * d + d + 4)  # BF16 K, FP8 V and its scale, per token
    if case["kind"] == "quant":
        n = case["tokens"]
        per = kv * (2 * d + d + 4) + (kv * 4 * d if case["with_k"] else 0)
        return {"bytes": case["layers"] * n * per + 4 * n, "flops": 0}
    if case["kind"] == "fill":
        n = sum(_lengths(case))
        return {"bytes": case["layers"] * n * (kv * 4 * d + page) + 4 * n, "flops": 0}
    s, layers = case["rows"], case.get("layers", 1)
    nbytes = flops = 0
    for t in _lengths(case):
        nbytes += t * page + 4 * s * h * d
        if case["kind"] != "op":
            nbytes += 4 * -(-t // _BLOCK)
        if case["kind"] in ("step", "prefill"):
            nbytes += s * kv * 4 * d  # the new K and V; their pages count among the context's
        flops += 4 * h * d * _visible(t, s)
    return {"bytes": layers * nbytes, "flops": layers * flops}


def tolerance(case):
    # codes, scales and the K copy are defined to the bit
    if case["kind"] in ("quant", "fill"):
        return "exact"
    # scores, probabilities, dequantized V and outputs in BF16: 3e-3 to 7e-3 off 64 bits
    return {"rel": 1e-2, "max": 0.1}


# ---------------------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(shape, g):
    return torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)


def _values(shape, g):
    """V: N(0, 1) with 1% of the (KV head, dimension) channels twenty times as large."""
    v = torch.randn(shape, generator=g, device="cuda")
    channels = shape[-2] * shape[-1]
    factor = torch.ones(channels, device="cuda")
    factor[torch.randperm(channels, generator=g, device="cuda")[: max(1, round(0.01 * channels))]] = 20.0
    return (v * factor.reshape(shape[-2:])).to(torch.bfloat16)


def _inputs(case, seed):
    """Everything a case starts from, from the seed alone: per layer the packed K and V of all
    sequences, and the queries (layer, sequence, row, head, dimension)."""
    g = _generator(seed)
    kv, d = case["kv"], case["dim"]
    if case["kind"] == "quant":
        v = _values((case["layers"], case["tokens"], kv, d), g)
        zero = torch.randperm(case["layers"] * case["tokens"], generator=g, device="cuda")
        v.view(-1, kv, d)[zero[: max(1, zero.numel() // 1000)]] = 0.0  # padding rows
        return {"k": _randn(tuple(v.shape), g), "v": v}
    total = sum(_lengths(case))
    layers = case.get("layers", 1)
    x = {"k": [_randn((total, kv, d), g) for _ in range(layers)], "v": [_values((total, kv, d), g) for _ in range(layers)]}
    if case["kind"] != "fill":
        x["q"] = _randn((layers, case["batch"], case["rows"], case["heads"], d), g)
    return x


def _codes(v):
    """(E4M3FN payload, fp32 scale) of BF16 V, one scale per token and KV head: max|v| / 448."""
    m = v.float().abs().amax(-1, keepdim=True)
    scale = m / torch.full_like(m, 448.0)
    scale = torch.where(scale == 0, torch.ones_like(scale), scale)
    return (v.float() / scale).to(torch.float8_e4m3fn), scale


def _new_rows(x, lengths, s):
    """Rows of the packed (total, KV, D) that are the last s tokens of every sequence: (B, s, KV, D)."""
    out, end = [], 0
    for t in lengths:
        end += t
        out.append(x[end - s:end])
    return torch.stack(out)


def prepare(case, seed):
    x = _inputs(case, seed)
    kv, d, kind = case["kv"], case["dim"], case["kind"]
    if kind == "quant":
        # a pool of its own whose blocks lie scattered
        cache = PagedKVCache(kv, d, num_layers=case["layers"], capacity_tokens=case["tokens"], seed=seed)
        cache.reserve(0, case["tokens"])
        return {"kind": kind, "cache": cache, "slots": cache.slot_mapping([0], case["tokens"]), "v": x["v"],
                "k": x["k"] if case["with_k"] else None}
    lengths = _lengths(case)
    if kind == "op":
        shape = (case["batch"], lengths[0], kv, d)
        payload, scale = _codes(x["v"][0].view(shape).transpose(1, 2).contiguous())
        return {"kind": kind, "q": x["q"][0].transpose(1, 2).contiguous(),
                "k": x["k"][0].view(shape).transpose(1, 2).contiguous(), "v": (payload, scale)}
    blocks = sum(-(-t // _BLOCK) for t in lengths)
    cache = PagedKVCache(kv, d, num_layers=case.get("layers", 1), batch=case["batch"], num_blocks=blocks + 8, seed=seed)
    if kind == "fill":
        return {"kind": kind, "cache": cache, "k": x["k"], "v": x["v"], "lengths": lengths}
    slots = None
    for layer, (k, v) in enumerate(zip(x["k"], x["v"])):
        slots = cache.prefill(layer, k, v, lengths, slots)
    if kind == "attend":
        q = x["q"].transpose(2, 3).contiguous()
        pages = (cache.k_pages, cache.v_pages, cache.v_scales)
        if case["layers"] == 1:
            q, pages = q[0], cache.layer(0)
        return {"kind": kind, "q": q, "pages": pages, "table": cache.block_table(), "lens": cache.seq_lens_tensor(),
                "longest": max(lengths), "cache": cache}
    # the context stands but for the new tokens, which each pass writes again
    s = case["rows"]
    state = {"kind": kind, "cache": cache, "starts": [t - s for t in lengths], "q": list(x["q"]),
             "k": [_new_rows(k, lengths, s) for k in x["k"]], "v": [_new_rows(v, lengths, s) for v in x["v"]]}
    if case.get("graph"):
        cache.reserve_all(max(lengths), q_heads=case["heads"], q_len=s)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _layers(state)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state["outputs"] = _layers(state)
        state["graph"] = graph
    return state


def _layers(state):
    cache, starts = state["cache"], state["starts"]
    return [cache.append_attend(layer, q, k, v, starts, q_token_major=True)
            for layer, (q, k, v) in enumerate(zip(state["q"], state["k"], state["v"]))]


def _pages(cache):
    return {"k_pages": cache.k_pages, "v_pages": cache.v_pages, "v_scales": cache.v_scales}


# ---------------------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind == "attend":
        kp, vp, vs = state["pages"]
        return ops.paged_attention(state["q"], kp, vp, vs, state["table"], state["lens"], state["longest"])
    if kind == "op":
        return ops.attention(state["q"], state["k"], state["v"], "hip")
    cache = state["cache"]
    if kind == "quant":
        ops.quant_append(state["v"], state["slots"], cache.k_pages, cache.v_pages, cache.v_scales, state["k"])
        return _pages(cache)
    if kind == "fill":
        slots = None
        for layer, (k, v) in enumerate(zip(state["k"], state["v"])):
            slots = cache.prefill(layer, k, v, state["lengths"], slots)
        return _pages(cache)
    if "graph" in state:
        state["graph"].replay()
        return {"out": state["outputs"], **_pages(cache)}
    return {"out": _layers(state), **_pages(cache)}


# ---------------------------------------------------------------------------- in 64 bits
def _attend64(q, k, v):
    """Softmax attention of q (s, H, D) over k and v (t, KV, D), all float64: (s, H, D)."""
    s, h, d = q.shape
    t, kv = k.shape[:2]
    group = h // kv
    hidden = torch.arange(t, device="cuda")[None, :] > torch.arange(t - s, t, device="cuda")[:, None]
    out = torch.empty_like(q)
    for head in range(h):
        scores = q[:, head].contiguous() @ k[:, head // group].t().contiguous() / math.sqrt(d)
        scores.masked_fill_(hidden, -math.inf)
        out[:, head] = torch.softmax(scores, -1) @ v[:, head // group].contiguous()
    return out


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    pages = {"k_pages": None, "v_pages": None, "v_scales": None}
    if kind in ("quant", "fill"):
        return None  # codes, copies and fp32 scales are defined to the bit: nothing is nearer than that
    lengths = _lengths(case)
    outs = []
    for layer, (k, v) in enumerate(zip(x["k"], x["v"])):
        payload, scale = _codes(v)
        v64, k64, rows, at = payload.double() * scale.double(), k.double(), [], 0
        for b, t in enumerate(lengths):
            rows.append(_attend64(x["q"][layer, b].double(), k64[at:at + t], v64[at:at + t]))
            at += t
        outs.append(torch.stack(rows))
    if kind in ("step", "prefill"):
        return {"out": outs, **pages}
    outs = [o.transpose(1, 2).contiguous() for o in outs]
    return outs[0] if kind == "op" or case["layers"] == 1 else torch.stack(outs)
