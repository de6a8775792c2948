"""What a user of this framework has it do, as cases that can be timed and checked.

A case is one step of a serving program, through the package's public entry points:

  decode          a token of every sequence: the batch uploaded, then append +
                  attention of each layer (KVPool.decode_append)
  prefill         chunks of prompts: the batch uploaded, then append + attention
                  of each layer (KVPool.prefill_append)
  q8              Q8_0 products of a layer, one call each (q8_matmul)
  model_decode    a whole decode step, logits out (Model.forward_decode_batch)
  model_prefill   a whole prefill of prompts, logits out (Model.forward_prefill)

Lengths are drawn from the case's own "lengths" number, so they are part of the
case; values, tokens, weights and page ids come from the seed.  K, V, q and
activations are N(0, 1), as they are behind a norm; weights are int8 of a normal
with a scale per block of 32 that keeps activations near 1.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

PAGE = 16
FULL_ROWS, LAST_BLOCK = 0, 1

# (query heads, K/V heads, head size)
HEADS_12X64 = {"heads": 12, "kv_heads": 12, "head_dim": 64}
HEADS_32X128 = {"heads": 32, "kv_heads": 32, "head_dim": 128}
HEADS_32_8X128 = {"heads": 32, "kv_heads": 8, "head_dim": 128}

MODEL_768 = {"dim": 768, "hidden": 2048, "layers": 12, "heads": 12, "kv_heads": 12, "vocab": 32000, "seq_len": 1024}
MODEL_2048 = {"dim": 2048, "hidden": 5632, "layers": 3, "heads": 32, "kv_heads": 4, "vocab": 32000, "seq_len": 2048}
MODEL_4096 = {"dim": 4096, "hidden": 11008, "layers": 2, "heads": 32, "kv_heads": 32, "vocab": 8000, "seq_len": 2048}


def listed():
    return [
        # one user generating: a token through a small model's twelve attention
        # layers, where latency and launches are everything
        {"name": "decode_1_ctx256", "kind": "decode", **HEADS_12X64, "layers": 12, "batch": 1, "shared": 0,
         "ctx_min": 256, "ctx_max": 256, "lengths": 0},
        # a serving batch of unequal contexts
        {"name": "decode_32_mixed", "kind": "decode", **HEADS_12X64, "layers": 12, "batch": 32, "shared": 0,
         "ctx_min": 16, "ctx_max": 1024, "lengths": 1},
        # users behind one cached system prompt of 512 tokens
        {"name": "decode_48_shared_prefix", "kind": "decode", **HEADS_12X64, "layers": 12, "batch": 48, "shared": 512,
         "ctx_min": 576, "ctx_max": 1024, "lengths": 2},
        # the largest decode: 64 long contexts, a K/V head per query head (one layer)
        {"name": "decode_64_ctx4096", "kind": "decode", **HEADS_32X128, "layers": 1, "batch": 64, "shared": 0,
         "ctx_min": 4096, "ctx_max": 4096, "lengths": 3},
        # grouped-query heads over retrieved documents of many lengths
        {"name": "decode_24_gqa", "kind": "decode", **HEADS_32_8X128, "layers": 2, "batch": 24, "shared": 0,
         "ctx_min": 512, "ctx_max": 8192, "lengths": 4},
        # eight fresh prompts through a small model's attention layers
        {"name": "prefill_8_prompts", "kind": "prefill", **HEADS_12X64, "layers": 12, "batch": 8, "cached_min": 0,
         "cached_max": 0, "new_min": 128, "new_max": 1024, "lengths": 5},
        # chunked prefill behind cached tokens, grouped-query heads
        {"name": "prefill_4_chunks_gqa", "kind": "prefill", **HEADS_32_8X128, "layers": 4, "batch": 4, "cached_min": 0,
         "cached_max": 4096, "new_min": 384, "new_max": 512, "lengths": 6},
        # prompts of a model whose head size is no power of two
        {"name": "prefill_6_head96", "kind": "prefill", "heads": 16, "kv_heads": 16, "head_dim": 96, "layers": 4,
         "batch": 6, "cached_min": 0, "cached_max": 0, "new_min": 50, "new_max": 700, "lengths": 7},
        # a feed-forward block's three products for one user
        {"name": "q8_ffn_1_row", "kind": "q8", "dim": 4096, "hidden": 11008, "rows": 1, "semantics": FULL_ROWS},
        # a whole decode step of a 110M-parameter model for a serving batch
        {"name": "model_decode_32", "kind": "model_decode", **MODEL_768, "batch": 32, "ctx_min": 448, "ctx_max": 576,
         "lengths": 8, "semantics": FULL_ROWS},
        # layers of a 7B-parameter model for a few users
        {"name": "model_decode_8_wide", "kind": "model_decode", **MODEL_4096, "batch": 8, "ctx_min": 900,
         "ctx_max": 1100, "lengths": 9, "semantics": FULL_ROWS},
        # the prompts of eight users through the 110M-parameter model: most products
        # of a program that answers long questions
        {"name": "model_prefill_8", "kind": "model_prefill", **MODEL_768, "batch": 8, "new_min": 128, "new_max": 1000,
         "lengths": 10, "semantics": FULL_ROWS},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_once(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "q8", "model_decode", "model_prefill"])
    lengths = rng.randrange(1 << 30)
    heads, kv_heads, head_dim = rng.choice(
        [(12, 12, 64), (12, 12, 64), (32, 32, 128), (32, 8, 128), (32, 8, 128), (32, 4, 64), (14, 2, 64),
         (16, 16, 96), (32, 32, 80), (16, 8, 256)])
    attention = {"kind": kind, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim,
                 "layers": rng.randint(1, 12), "lengths": lengths}
    if kind == "decode":
        top = _log_int(rng, 16, 8192)
        low = _log_int(rng, max(1, top // 16), top)
        shared = rng.choice([0, 0, 0, low // 2])
        return {**attention, "batch": _log_int(rng, 1, 64), "shared": shared, "ctx_min": max(low, shared + 1),
                "ctx_max": max(top, shared + 1)}
    if kind == "prefill":
        top = _log_int(rng, 16, 4096)
        cached = rng.choice([0, 0, _log_int(rng, 16, 4096)])
        return {**attention, "batch": _log_int(rng, 1, 16), "cached_min": cached // 4, "cached_max": cached,
                "new_min": _log_int(rng, max(1, top // 8), top), "new_max": top}
    semantics = rng.choice([FULL_ROWS, FULL_ROWS, FULL_ROWS, LAST_BLOCK])
    if kind == "q8":
        dim, hidden = rng.choice([(768, 2048), (2048, 5632), (4096, 11008), (4096, 11008), (4096, 14336), (1056, 2720)])
        return {"kind": kind, "dim": dim, "hidden": hidden, "rows": _log_int(rng, 1, 1024), "semantics": semantics}
    model = rng.choice([MODEL_768, MODEL_2048, MODEL_4096])
    if kind == "model_decode":
        top = _log_int(rng, 16, model["seq_len"])
        return {"kind": kind, **model, "batch": _log_int(rng, 1, 64), "ctx_min": _log_int(rng, max(1, top // 8), top),
                "ctx_max": top, "lengths": lengths, "semantics": semantics}
    top = _log_int(rng, 8, model["seq_len"])
    return {"kind": kind, **model, "batch": _log_int(rng, 1, 8), "new_min": _log_int(rng, max(1, top // 8), top),
            "new_max": top, "lengths": lengths, "semantics": semantics}


def draw(rng):
    while True:
        case = _draw_once(rng)
        w = work(case)
        if w["bytes"] <= 6e9 and w["flops"] <= (6e11 if case["kind"].startswith("model") else 3e11):
            return case


# ------------------------------------------------------------------ lengths

def _ints(case, low, high, salt=0):
    r = random.Random(case["lengths"] * 3 + salt)
    return [r.randint(low, high) for _ in range(case["batch"])]


def _contexts(case):
    """Keys that each sequence of a decode batch attends, the new one among them."""
    return _ints(case, case["ctx_min"], case["ctx_max"])


def _chunks(case):
    """(cached tokens, new tokens) of each sequence of a prefill batch."""
    cached = _ints(case, case["cached_min"], case["cached_max"], 1) if "cached_max" in case else [0] * case["batch"]
    return cached, _ints(case, case["new_min"], case["new_max"])


def _head_dim(case):
    return case["head_dim"] if "head_dim" in case else case["dim"] // case["heads"]


def _products(case):
    """(rows of W, columns of W) of each Q8 matrix of a layer."""
    d, h, kv = case["dim"], case["hidden"], case["kv_heads"] * _head_dim(case)
    return {"wq": (d, d), "wk": (kv, d), "wv": (kv, d), "wo": (d, d), "w1": (h, d), "w2": (d, h), "w3": (h, d)}


def _ffn_shapes(case):
    return [(case["hidden"], case["dim"]), (case["hidden"], case["dim"]), (case["dim"], case["hidden"])]


# --------------------------------------------------------------------- work

def _shared_pages(case):
    """Whole pages that every sequence of a decode batch shares (the newest row is its own)."""
    return case.get("shared", 0) // PAGE if case["batch"] > 1 else 0


def _attention_work(case, keys, rows, pairs):
    """One layer: `keys` K/V rows read, `rows` queries (each row's K/V written too), `pairs` query-key pairs."""
    q, kv = case["heads"] * _head_dim(case), case["kv_heads"] * _head_dim(case)
    return {"bytes": 8 * kv * (keys + rows) + 8 * q * rows, "flops": 4.0 * q * pairs}


def _q8_work(rows, d, n, semantics):
    cols = n if semantics == FULL_ROWS else 32
    return {"bytes": d * (cols // 32) * 36 + 4 * rows * (cols + d), "flops": 2.0 * rows * d * cols}


def work(case):
    kind = case["kind"]
    if kind == "q8":
        parts = [_q8_work(case["rows"], d, n, case["semantics"]) for d, n in _ffn_shapes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if kind.endswith("decode"):
        ctx = _contexts(case)
        rows, pairs, saved = len(ctx), sum(ctx), _shared_pages(case) * PAGE * (len(ctx) - 1)
        attention = _attention_work(case, pairs - saved, rows, pairs)
    else:
        cached, new = _chunks(case)
        rows = sum(new)
        pairs = sum(n * c + n * (n + 1) // 2 for c, n in zip(cached, new))
        attention = _attention_work(case, rows + sum(cached), rows, pairs)
    layers = case["layers"]
    total = {k: v * layers for k, v in attention.items()}
    if kind.startswith("model"):
        # beside attention: every weight read once, each row's embedding, the logits
        for d, n in _products(case).values():
            cols = n if case["semantics"] == FULL_ROWS else 32
            total["bytes"] += layers * d * (cols // 32) * 36
            total["flops"] += layers * 2.0 * rows * d * cols
        out_rows = case["batch"]
        total["bytes"] += 4 * case["vocab"] * case["dim"] + 4 * out_rows * case["vocab"] + 4 * rows * case["dim"]
        total["flops"] += 2.0 * out_rows * case["vocab"] * case["dim"]
    return total


# ------------------------------------------------------------------- inputs

def _generator(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + salt)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _tables(need, shared, pages, seed):
    """Block tables [batch][most pages]: `shared` first pages common to all, the rest taken in turn
    from one permutation of the pool."""
    order = np.random.default_rng(int(seed)).permutation(pages).astype(np.int32)
    tables = np.zeros((len(need), max(need)), np.int32)
    tables[:, :shared] = order[:shared]
    at = shared
    for b, n in enumerate(need):
        tables[b, shared:n] = order[at:at + n - shared]
        at += n - shared
    return tables


def _pool_pages(need, shared):
    used = shared + sum(n - shared for n in need)
    return used + used // 8 + 3  # a pool has spare pages


def _attention_inputs(case, seed):
    """Everything before the pool handle: K/V pools [pages][layers][16][kv_dim], tables, and per layer q, k, v."""
    head_dim = _head_dim(case)
    q_dim, kv_dim = case["heads"] * head_dim, case["kv_heads"] * head_dim
    if case["kind"].endswith("decode"):
        ctx = _contexts(case)
        need, shared, rows = [-(-c // PAGE) for c in ctx], _shared_pages(case), len(ctx)
        s = {"positions": np.array(ctx, np.int32) - 1}
    else:
        cached, new = _chunks(case)
        need, shared, rows = [-(-(c + n) // PAGE) for c, n in zip(cached, new)], 0, sum(new)
        s = {"start": np.array(cached, np.int32), "count": np.array(new, np.int32)}
    pages, layers, g = _pool_pages(need, shared), case["layers"], _generator(seed)
    s["tables"] = _tables(need, shared, pages, seed)
    s["k_pool"] = _normal(g, pages, layers, PAGE, kv_dim)
    s["v_pool"] = _normal(g, pages, layers, PAGE, kv_dim)
    if not case["kind"].startswith("model"):
        s["q"] = _normal(g, layers, rows, q_dim)
        s["k"] = _normal(g, layers, rows, kv_dim)
        s["v"] = _normal(g, layers, rows, kv_dim)
    else:
        s["tokens"] = np.random.default_rng(int(seed) + 1).integers(0, case["vocab"], rows).astype(np.int32)
    return s


def _q8_values(g, rows, cols):
    """Scales [rows][cols/32] and int8 weights [rows][cols/32][32] whose products keep activations near 1."""
    q = _normal(g, rows, cols // 32, 32).mul_(42.0).round_().clamp_(-127, 127).to(torch.int8)
    scale = (torch.rand(rows, cols // 32, generator=g, device="cuda") * 0.5 + 0.75) / (42.0 * math.sqrt(cols))
    return scale, q


def _q8_bytes(scale, q):
    """BlockQ8 rows: per 32 weights a float scale and 32 int8, 36 bytes."""
    return torch.cat((scale.unsqueeze(-1).contiguous().view(torch.uint8), q.view(torch.uint8)), dim=-1).reshape(-1)


def _q8_inputs(case, seed):
    g = _generator(seed)
    return [(_q8_values(g, d, n), _normal(g, case["rows"], n)) for d, n in _ffn_shapes(case)]


def _model_weights(case, seed):
    g, layers, dim = _generator(seed, 1), case["layers"], case["dim"]
    w = {"emb": _normal(g, case["vocab"], dim),
         "rms_att": torch.rand(layers, dim, generator=g, device="cuda") + 0.5,
         "rms_ffn": torch.rand(layers, dim, generator=g, device="cuda") + 0.5,
         "rms_final": torch.rand(dim, generator=g, device="cuda") + 0.5}
    for name, (d, n) in _products(case).items():
        w[name] = _q8_values(g, layers * d, n)
    half = _head_dim(case) // 2
    angle = np.arange(case["seq_len"])[:, None] * 10000.0 ** (-np.arange(half)[None, :] / half)
    w["cos"], w["sin"] = np.cos(angle).astype(np.float32), np.sin(angle).astype(np.float32)
    return w


def _model_file(case, w):
    """The model file: header, then the sections in its order."""
    header = np.array([case[k] for k in ("dim", "hidden", "layers", "heads", "kv_heads", "vocab", "seq_len")], np.int32)
    sections = [header.view(np.uint8)]
    for name in ("emb", "rms_att", "wq", "wk", "wv", "wo", "rms_ffn", "w1", "w2", "w3", "rms_final", "cos", "sin"):
        v = w[name]
        if isinstance(v, tuple):
            v = _q8_bytes(*v)
        if isinstance(v, torch.Tensor):
            v = v.cpu().numpy()
        sections.append(np.ascontiguousarray(v).reshape(-1).view(np.uint8))
    return np.concatenate(sections)


def prepare(case, seed):
    import nitrorag_amd as na

    if case["kind"] == "q8":
        ops = []
        for (scale, q), x in _q8_inputs(case, seed):
            ops.append((_q8_bytes(scale, q), x, torch.empty(x.shape[0], q.shape[0], device="cuda")))
        return {"case": case, "ops": ops}
    s = _attention_inputs(case, seed)
    s["case"] = case
    s["pool"] = na.KVPool.wrap(s["k_pool"], s["v_pool"])
    if case["kind"].startswith("model"):
        s["model"] = na.Model(_model_file(case, _model_weights(case, seed)))
        s["logits"] = torch.empty(case["batch"], case["vocab"], device="cuda")
    else:
        s["out"] = torch.empty_like(s["q"])
    return s


# ---------------------------------------------------------------------- run

def run(s):
    import nitrorag_amd as na

    case = s["case"]
    if case["kind"] == "q8":
        for w, x, out in s["ops"]:
            na.q8_matmul(w, x, out, case["semantics"])
        return [out for _, _, out in s["ops"]]
    pool = s["pool"]
    if case["kind"].endswith("decode"):
        pool.upload_decode_batch(s["tables"], s["positions"])
    else:
        pool.upload_prefill_batch(s["tables"], s["start"], s["count"])
    if case["kind"] == "model_decode":
        s["model"].forward_decode_batch(pool, s["tokens"], s["logits"], case["semantics"])
        return s["logits"], s["k_pool"], s["v_pool"]
    if case["kind"] == "model_prefill":
        s["model"].forward_prefill(pool, s["tokens"], s["logits"], case["semantics"])
        return s["logits"], s["k_pool"], s["v_pool"]
    step = pool.decode_append if case["kind"] == "decode" else pool.prefill_append
    shape = (case["heads"], case["kv_heads"], case["head_dim"])
    for layer in range(case["layers"]):
        step(layer, s["q"][layer], s["k"][layer], s["v"][layer], s["out"][layer], *shape)
    return s["out"], s["k_pool"], s["v_pool"]


# -------------------------------------------------------------------- exact

def _slots(s):
    """Per sequence: the pool slots of its keys, its first new key, its first row in the batch."""
    if "positions" in s:
        spans = [(int(p), 1) for p in s["positions"]]
    else:
        spans = [(int(c), int(n)) for c, n in zip(s["start"], s["count"])]
    row = 0
    for b, (first, count) in enumerate(spans):
        at = np.arange(first + count)
        slots = s["tables"][b][at // PAGE].astype(np.int64) * PAGE + at % PAGE
        yield torch.from_numpy(slots).cuda(), first, count, row
        row += count


def _attend(case, s, layer, q, k, v):
    """Appends k, v (64-bit rows) to the pools of `layer` and attends, in 64 bits."""
    heads, kv_heads, head_dim = case["heads"], case["kv_heads"], _head_dim(case)
    out = torch.empty(q.shape[0], heads * head_dim, device="cuda", dtype=torch.float64)
    pools = [s["k_pool"], s["v_pool"]]
    rows = list(_slots(s))
    for slots, first, count, row in rows:
        for pool, new in zip(pools, (k, v)):
            mine = slots[first:]
            pool[mine // PAGE, layer, mine % PAGE] = new[row:row + count].to(pool.dtype)
    for slots, first, count, row in rows:
        keys, values = (p[slots // PAGE, layer, slots % PAGE].double().view(-1, kv_heads, head_dim) for p in pools)
        if k.dtype == torch.float64:  # this step's rows without the pool's rounding
            keys[first:] = k[row:row + count].view(count, kv_heads, head_dim)
            values[first:] = v[row:row + count].view(count, kv_heads, head_dim)
        mine = q[row:row + count].double().view(count, heads, head_dim)
        seen = torch.arange(first + count, device="cuda")[None, :] <= first + torch.arange(count, device="cuda")[:, None]
        for h in range(heads):
            kh = h * kv_heads // heads
            score = mine[:, h] @ keys[:, kh].T / math.sqrt(head_dim)
            weight = torch.softmax(score.masked_fill(~seen, -math.inf), dim=-1)
            out[row:row + count, h * head_dim:(h + 1) * head_dim] = weight @ values[:, kh]
    return out


def _q8_product(case, scale, q, x):
    w = q.double() * scale.double().unsqueeze(-1)
    w = w.reshape(w.shape[0], -1)
    if case["semantics"] == LAST_BLOCK:
        w, x = w[:, -32:], x[:, -32:]
    return x.double() @ w.T


def _rms_norm(x, weight):
    return weight.double() * x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-5)


def _rotate(x, cos, sin, head_dim):
    pairs = x.view(x.shape[0], -1, head_dim // 2, 2)
    a, b, c, d = pairs[..., 0], pairs[..., 1], cos[:, None, :], sin[:, None, :]
    return torch.stack((a * c - b * d, a * d + b * c), dim=-1).reshape(x.shape)


def _exact_model(case, seed):
    s, w = _attention_inputs(case, seed), _model_weights(case, seed)
    if "positions" in s:
        at, last = s["positions"], np.arange(case["batch"])
    else:
        at = np.concatenate([np.arange(c, c + n) for c, n in zip(s["start"], s["count"])])
        last = np.cumsum(s["count"]) - 1
    cos, sin = (torch.from_numpy(w[n][at]).cuda().double() for n in ("cos", "sin"))
    x = w["emb"][torch.from_numpy(s["tokens"].astype(np.int64)).cuda()].double()
    shapes, head_dim = _products(case), _head_dim(case)
    for layer in range(case["layers"]):
        def product(name, v):
            d = shapes[name][0]
            scale, q = (t[layer * d:(layer + 1) * d] for t in w[name])
            return _q8_product(case, scale, q, v)

        y = _rms_norm(x, w["rms_att"][layer])
        q, k = (_rotate(product(n, y), cos, sin, head_dim) for n in ("wq", "wk"))
        x = x + product("wo", _attend(case, s, layer, q, k, product("wv", y)))
        y = _rms_norm(x, w["rms_ffn"][layer])
        gate = product("w1", y)
        x = x + product("w2", gate * torch.sigmoid(gate) * product("w3", y))
    logits = _rms_norm(x[torch.from_numpy(last).cuda()], w["rms_final"]) @ w["emb"].double().T
    return logits, s["k_pool"], s["v_pool"]


def exact(case, seed):
    """run()'s outputs in 64 bits, from plain torch (pools: their rows as stored, in 32 bits)."""
    if case["kind"] == "q8":
        return [_q8_product(case, scale, q, x) for (scale, q), x in _q8_inputs(case, seed)]
    if case["kind"].startswith("model"):
        return _exact_model(case, seed)
    s = _attention_inputs(case, seed)
    out = torch.stack([_attend(case, s, i, s["q"][i], s["k"][i], s["v"][i]) for i in range(case["layers"])])
    return out, s["k_pool"], s["v_pool"]


def tolerance(case):
    """About four times what the outputs measure against exact(): 32-bit sums everywhere, except that
    prefill attention at head sizes 32, 64 and 128 holds V and the weights to 16 significant bits."""
    kind = case["kind"]
    if kind in ("decode", "q8"):
        return {"rel": 1e-6}
    if kind == "model_decode":
        return {"rel": 2.5e-6}
    if kind == "model_prefill":
        return {"rel": 9e-5}
    return {"rel": 7e-5 if case["head_dim"] in (32, 64, 128) else 1.5e-6}
