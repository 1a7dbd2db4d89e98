"""What a program built on this library has it do, as timed cases.

Every case goes through the public Python faces (FactorLayer, FactorSet,
GpuContext, SageDecodeState, DecoderBlock, LmHead and the trunk functions).
Shapes come from the repository's configurations (config 1: a 4096 x 4096
layer of rank 1024; config 2: that layer as a GEMM; config 3: the seven
projections of a 4096-wide decoder block at 0.55 bit a weight; config 4:
attention of 32 heads over 4096 tokens; config 5: a model of such blocks with
a 128256-row head) or are generic.  Inputs are made from the seed alone.
"""
import math

import numpy as np
import torch

import quantibbler_amd as qa
from quantibbler_amd.gpu import FactorSet, embed, rms_norm_dev

DEV = "cuda"
THETA, EPS = 500000.0, 1e-5

# d, heads, kv heads, head dim, ffn: config 3's block and a smaller one
GEOMETRY = {"wide": (4096, 32, 8, 128, 14336), "narrow": (2048, 16, 8, 128, 5632)}


def listed():
    return [
        # config 1: one projection of a decode step, the smallest call; its latency is the launches'
        {"name": "linear-token", "kind": "linear", "m": 4096, "n": 4096, "r": 1024, "batch": 1, "y": "bfloat16",
         "bias": False},
        # a small layer with a bias, no size a multiple of a tile, at a short prompt's batch
        {"name": "linear-ragged", "kind": "linear", "m": 1000, "n": 1537, "r": 301, "batch": 37, "y": "float32",
         "bias": True},
        # config 2: the layer over a prompt's 2048 tokens
        {"name": "linear-prefill", "kind": "linear", "m": 4096, "n": 4096, "r": 1024, "batch": 2048, "y": "bfloat16",
         "bias": False},
        # config 3: the projections of a decoded token, blocks decoded as one set
        {"name": "set-token", "kind": "set", "geometry": "wide", "blocks": 2, "batch": 1},
        # config 4: causal block-scaled attention of a whole prompt
        {"name": "sage-prompt", "kind": "sage_blk", "batch": 1, "heads": 32, "kv_heads": 32, "seq": 4096,
         "causal": True},
        # the reference scheme (f32 operands) over a prompt that ends inside a block, grouped heads
        {"name": "sage-reference", "kind": "sage_ref", "batch": 1, "heads": 16, "kv_heads": 8, "seq": 1999, "d": 128,
         "causal": True, "block": 64},
        # one decode step of the reference scheme on a kept state, config 3's heads
        {"name": "sage-step", "kind": "sage_step", "heads": 32, "kv_heads": 8, "d": 128, "seq": 4090, "block": 64},
        # the exact f32 face: a query chunk against a longer key range
        {"name": "attention-exact", "kind": "exact", "batch": 1, "heads": 16, "kv_heads": 8, "seq_q": 777,
         "seq_kv": 1300, "d": 128, "causal": True},
        # a decoder block at fp32 serving on the exact attention face, one token
        {"name": "block-token-fp32", "kind": "decode", "geometry": "wide", "context": 700, "batch": 1,
         "serving": "fp32", "face": "exact"},
        # a decoder block stepping 32 sequences of different lengths (batched serving)
        {"name": "block-batch", "kind": "decode", "geometry": "wide", "context": 2085, "batch": 32,
         "serving": "bf16", "face": "sage"},
        # a decoder block over a prompt of 2048 tokens (the largest)
        {"name": "block-prompt", "kind": "prefill", "geometry": "wide", "tokens": 2048},
        # a whole greedy-decode call of a cut-down config 5: embedding, blocks, final norm, logits
        {"name": "model-token", "kind": "model", "geometry": "wide", "blocks": 2, "context": 2085, "vocab": 128256},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "set", "sage_blk", "sage_ref", "sage_step", "exact", "decode",
                       "decode", "prefill", "model"])
    if kind == "linear":
        m, n = _log(rng, 200, 14336), _log(rng, 200, 14336)
        if rng.random() < 0.6:  # widths are mostly multiples of a wave
            m, n = max(256, m // 128 * 128), max(256, n // 128 * 128)
        r = max(16, min(_rank(m, n), 1800))
        batch = min(_log(rng, 1, 4096), int(1.4e11 / (2 * r * (m + n))))
        return {"kind": kind, "m": m, "n": n, "r": r, "batch": max(1, batch),
                "y": rng.choice(["bfloat16", "float32"]), "bias": rng.random() < 0.3}
    if kind == "set":
        return {"kind": kind, "geometry": rng.choice(["wide", "narrow"]), "blocks": rng.randint(1, 2),
                "batch": _log(rng, 1, 32)}
    if kind == "sage_blk":
        kv = rng.choice([2, 4, 8])
        return {"kind": kind, "batch": rng.randint(1, 2), "heads": kv * rng.choice([1, 2, 4]), "kv_heads": kv,
                "seq": _log(rng, 100, 4096), "causal": rng.random() < 0.7}
    if kind == "sage_ref":
        kv = rng.choice([2, 4, 8])
        return {"kind": kind, "batch": 1, "heads": kv * rng.choice([1, 2]), "kv_heads": kv, "seq": _log(rng, 60, 1900),
                "d": rng.choice([64, 128]), "causal": rng.random() < 0.7, "block": rng.choice([32, 64, 128])}
    if kind == "sage_step":
        kv = rng.choice([2, 4, 8])
        return {"kind": kind, "heads": kv * rng.choice([1, 2, 4]), "kv_heads": kv, "d": rng.choice([64, 128]),
                "seq": _log(rng, 100, 8000), "block": rng.choice([32, 64])}
    if kind == "exact":
        kv = rng.choice([2, 4, 8])
        skv = _log(rng, 60, 1300)
        return {"kind": kind, "batch": rng.randint(1, 2), "heads": kv * rng.choice([1, 2]), "kv_heads": kv,
                "seq_q": min(skv, _log(rng, 1, 777)), "seq_kv": skv, "d": rng.choice([64, 80, 128]),
                "causal": rng.random() < 0.7}
    geometry = rng.choice(["wide", "narrow"])
    if kind == "decode":
        if rng.random() < 0.3:
            return {"kind": kind, "geometry": geometry, "context": _log(rng, 30, 2085), "batch": 1, "serving": "fp32",
                    "face": rng.choice(["exact", "sage"])}
        return {"kind": kind, "geometry": geometry, "context": _log(rng, 30, 2085), "batch": _log(rng, 1, 32),
                "serving": "bf16", "face": "sage"}
    if kind == "prefill":
        return {"kind": kind, "geometry": geometry, "tokens": _log(rng, 10, 2048)}
    return {"kind": kind, "geometry": geometry, "blocks": rng.randint(1, 2), "context": _log(rng, 30, 2085),
            "vocab": _log(rng, 8000, 128256)}


# ---- inputs ------------------------------------------------------------------

def _rank(m, n):
    """The rank that spends 0.55 bit a weight on an m x n layer, scales in 16 bits."""
    return int(round((0.55 * m * n - 16 * (2 * m + n)) / (m + n)))


def _normal(seed, tag, shape, dtype=torch.float32):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + int(tag))
    return torch.randn(shape, device=DEV, generator=g, dtype=dtype)


def _parts(seed, tag, m, n, r, bias=False):
    """A layer's fields as a loader hands them over: packed signs, scales that are fp16 values, maybe a bias."""
    rng = np.random.default_rng([int(seed), int(tag)])
    ub = np.frombuffer(rng.bytes(m * ((r + 7) // 8)), np.uint8).reshape(m, -1)
    vt = np.frombuffer(rng.bytes(r * ((n + 7) // 8)), np.uint8).reshape(r, -1)
    s1 = (np.exp(0.3 * rng.standard_normal(m)) / math.sqrt(r * n)).astype(np.float16).astype(np.float32)
    s2 = np.exp(0.3 * rng.standard_normal(n)).astype(np.float16).astype(np.float32)
    b = rng.standard_normal(m).astype(np.float32) if bias else None
    return m, n, r, ub, vt, s1, s2, b


def _layer(ctx, parts):
    m, n, r, ub, vt, s1, s2, b = parts
    return qa.FactorLayer.from_rows(ctx, m, n, r, ub, vt, s1, s2, b)


def _block_shapes(geometry):
    d, H, Hk, hd, ffn = GEOMETRY[geometry]
    return [(H * hd, d), (Hk * hd, d), (Hk * hd, d), (d, H * hd), (ffn, d), (ffn, d), (d, ffn)]


def _block_parts(seed, block, geometry):
    return [_parts(seed, 100 * block + i, m, n, _rank(m, n)) for i, (m, n) in enumerate(_block_shapes(geometry))]


def _norm_weights(seed, block, d):
    rng = np.random.default_rng([int(seed), 7000 + block])
    return [(1.0 + 0.1 * rng.standard_normal(d)).astype(np.float16).astype(np.float32) for _ in range(2)]


def _bytes(n):
    return torch.empty(max(int(n), 16), dtype=torch.uint8, device=DEV)


class _Address:
    """A device address of a block's as an array that torch can view (the view keeps the block)."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (int(ptr), False),
                                         "version": 2}


def _caches(block, geometry):
    _, _, Hk, hd, _ = GEOMETRY[geometry]
    return [torch.as_tensor(_Address(block, p, (block.n_seqs, block.capacity, Hk * hd)), device=DEV)
            for p in block.cache_ptrs()]


def _cached_rows(seed, block, n_seqs, rows, width):
    """Keys with a channel mean, as trained models have, and values."""
    k = _normal(seed, 8000 + block, (n_seqs, rows, width)) + 2.0 * _normal(seed, 8100 + block, (1, 1, width))
    return k, _normal(seed, 8200 + block, (n_seqs, rows, width))


def _contexts(case):
    """The cached lengths of a batched step's sequences: from half the context to all of it."""
    n, c = case.get("batch", 1), case["context"]
    return [c - (i * (c // 2)) // n for i in range(n)]


def _make_block(ctx, seed, index, case, n_seqs, capacity):
    geometry = case["geometry"]
    d, H, Hk, hd, _ = GEOMETRY[geometry]
    layers = [_layer(ctx, p) for p in _block_parts(seed, index, geometry)]
    w_in, w_post = _norm_weights(seed, index, d)
    block = qa.DecoderBlock(ctx, layers, w_in, w_post, H, Hk, hd, THETA, EPS, capacity, n_seqs=n_seqs)
    block.set_attention_face(case.get("face", "sage"))
    block.set_serving(case.get("serving", "bf16"))
    return block


def _fill(block, seed, index, case, contexts):
    _, _, Hk, hd, _ = GEOMETRY[case["geometry"]]
    for cache, rows in zip(_caches(block, case["geometry"]),
                           _cached_rows(seed, index, len(contexts), max(contexts), Hk * hd)):
        cache[:, :max(contexts)].copy_(rows)
    block.set_filled(contexts)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["kind"]](state)


def _prepare_linear(case, seed):
    ctx = qa.GpuContext(0)
    layer = _layer(ctx, _parts(seed, 1, case["m"], case["n"], case["r"], case["bias"]))
    need = layer.workspace_size(case["batch"])
    y = torch.empty((case["batch"], case["m"]), dtype=getattr(torch, case["y"]), device=DEV)
    return dict(case, ctx=ctx, layer=layer, x=_linear_x(case, seed), out=y, need=need, ws=_bytes(need),
                stream=torch.cuda.current_stream())


def _linear_x(case, seed):
    scale = torch.exp(0.5 * _normal(seed, 2, (1, case["n"])))  # channels of unlike size, as activations have
    return (_normal(seed, 3, (case["batch"], case["n"])) * scale).to(torch.bfloat16)


def _run_linear(s):
    s["layer"].linear_dev(s["x"], s["batch"], s["out"], s["y"], s["ws"], s["need"], s["stream"])
    return s["out"]


def _prepare_set(case, seed):
    ctx = qa.GpuContext(0)
    parts = [p for b in range(case["blocks"]) for p in _block_parts(seed, b, case["geometry"])]
    layers = FactorSet(ctx, [_layer(ctx, p) for p in parts])
    n = case["batch"]
    x = _normal(seed, 3, (n * sum(p[1] for p in parts),)).to(torch.bfloat16)
    y = torch.empty(n * sum(p[0] for p in parts), dtype=torch.bfloat16, device=DEV)
    need = layers.workspace_size() if n == 1 else layers.workspace_size_batch(n)
    return dict(case, ctx=ctx, set=layers, x=x, y=y, need=need, ws=_bytes(need), stream=torch.cuda.current_stream())


def _run_set(s):
    if s["batch"] == 1:
        s["set"].decode_dev(s["x"], s["y"], s["ws"], s["need"], s["stream"])
    else:
        s["set"].decode_batch_dev(s["batch"], s["x"], s["y"], s["ws"], s["need"], s["stream"])
    return s["y"]


def _attention_inputs(seed, b, h, hk, sq, skv, d, dtype):
    q = _normal(seed, 1, (b, h, sq, d))
    k = _normal(seed, 2, (b, hk, skv, d)) + 2.0 * _normal(seed, 3, (b, hk, 1, d))
    v = _normal(seed, 4, (b, hk, skv, d))
    return q.to(dtype), k.to(dtype), v.to(dtype)


def _prepare_sage_blk(case, seed):
    ctx = qa.GpuContext(0)
    b, h, hk, s = case["batch"], case["heads"], case["kv_heads"], case["seq"]
    q, k, v = _attention_inputs(seed, b, h, hk, s, s, 128, torch.bfloat16)
    shape = qa.AttentionShape(b, h, hk, s, s, 128, 128)
    need = ctx.sage_blk_workspace_size(shape)
    return dict(case, ctx=ctx, shape=shape, q=q, k=k, v=v, out=torch.empty_like(q), need=need, ws=_bytes(need),
                stream=torch.cuda.current_stream())


def _run_sage_blk(s):
    s["ctx"].attention_sage_blk_dev(s["shape"], s["q"], s["k"], s["v"], s["causal"], s["out"], s["ws"], s["need"],
                                    s["stream"])
    return s["out"]


def _prepare_sage_ref(case, seed):
    ctx = qa.GpuContext(0)
    b, h, hk, s, d = case["batch"], case["heads"], case["kv_heads"], case["seq"], case["d"]
    q, k, v = _attention_inputs(seed, b, h, hk, s, s, d, torch.float32)
    return dict(case, ctx=ctx, shape=qa.AttentionShape(b, h, hk, s, s, d, d), q=q, k=k, v=v, out=torch.empty_like(q),
                stream=torch.cuda.current_stream())


def _run_sage_ref(s):
    s["ctx"].attention_sage_dev(s["shape"], s["q"], s["k"], s["v"], s["causal"], s["block"], s["out"], s["stream"])
    return s["out"]


def _step_inputs(case, seed):
    h, hk, s, d = case["heads"], case["kv_heads"], case["seq"], case["d"]
    q = _normal(seed, 1, (h, d))
    k = _normal(seed, 2, (s, hk, d)) + 2.0 * _normal(seed, 3, (1, hk, d))
    return q, k, _normal(seed, 4, (s, hk, d))


def _prepare_sage_step(case, seed):
    ctx = qa.GpuContext(0)
    h, hk, s, d, block = case["heads"], case["kv_heads"], case["seq"], case["d"], case["block"]
    q, k, v = _step_inputs(case, seed)
    state = qa.SageDecodeState(ctx, h, hk, d, d, s, block, _bytes(qa.SageDecodeState.size(ctx, h, hk, d, d, s, block)))
    out = torch.empty((h, d), dtype=torch.float32, device=DEV)
    stream = torch.cuda.current_stream()
    if s > 1:  # the loop's earlier steps have left the codes of the rows before this one
        state.step(q, k, v, s - 1, out, stream)
    return dict(case, ctx=ctx, state=state, q=q, k=k, v=v, out=out, stream=stream)


def _run_sage_step(s):
    s["state"].tokens = s["seq"] - 1  # the step that appended the last row
    s["state"].step(s["q"], s["k"], s["v"], s["seq"], s["out"], s["stream"])
    return s["out"]


def _prepare_exact(case, seed):
    ctx = qa.GpuContext(0)
    b, h, hk, sq, skv, d = (case[x] for x in ("batch", "heads", "kv_heads", "seq_q", "seq_kv", "d"))
    q, k, v = _attention_inputs(seed, b, h, hk, sq, skv, d, torch.float32)
    return dict(case, ctx=ctx, shape=qa.AttentionShape(b, h, hk, sq, skv, d, d), q=q, k=k, v=v,
                out=torch.empty_like(q), stream=torch.cuda.current_stream())


def _run_exact(s):
    s["ctx"].attention_dev(s["shape"], s["q"], s["k"], s["v"], s["causal"], s["out"], s["stream"])
    return s["out"]


def _prepare_decode(case, seed):
    ctx = qa.GpuContext(0)
    n, contexts = case["batch"], _contexts(case)
    d = GEOMETRY[case["geometry"]][0]
    block = _make_block(ctx, seed, 0, case, n, case["context"] + 1)
    _fill(block, seed, 0, case, contexts)
    need = block.decode_batch_workspace_size(n) if n > 1 else 0
    state = dict(case, ctx=ctx, block=block, contexts=contexts, h0=_normal(seed, 3, (n, d)),
                 h=torch.empty((n, d), dtype=torch.float32, device=DEV), need=need, ws=_bytes(need),
                 caches=_caches(block, case["geometry"]), rows=torch.arange(n, device=DEV),
                 at=torch.tensor(contexts, device=DEV), stream=torch.cuda.current_stream())
    _run_decode(state)  # the attention state's codes of the cached rows, as the loop's earlier steps leave them
    return state


def _run_decode(s):
    block = s["block"]
    s["h"].copy_(s["h0"])  # the block before this one writes its rows here
    if "state_ready" in s:
        block.set_positions(s["contexts"])  # the state is stepped through the rows before this token
    s["state_ready"] = True
    if s["batch"] == 1:
        block.decode_dev(s["h"], s["contexts"][0], s["stream"])
    else:
        block.decode_batch_dev(s["h"], s["contexts"], s["ws"], s["need"], s["stream"])
    return [s["h"]] + [c[s["rows"], s["at"]] for c in s["caches"]]


def _prepare_prefill(case, seed):
    ctx = qa.GpuContext(0)
    n, d = case["tokens"], GEOMETRY[case["geometry"]][0]
    block = _make_block(ctx, seed, 0, case, 1, n)
    need = block.prefill_workspace_size(n)
    return dict(case, ctx=ctx, block=block, h0=_normal(seed, 3, (n, d)),
                h=torch.empty((n, d), dtype=torch.float32, device=DEV), need=need, ws=_bytes(need),
                caches=_caches(block, case["geometry"]), stream=torch.cuda.current_stream())


def _run_prefill(s):
    s["h"].copy_(s["h0"])
    s["block"].prefill_dev(s["h"], s["tokens"], s["ws"], s["need"], s["stream"])
    return [s["h"]] + s["caches"]


def _model_tables(seed, case):
    vocab, d = case["vocab"], GEOMETRY[case["geometry"]][0]
    table = _normal(seed, 5, (vocab, d)).to(torch.bfloat16).to(torch.float32)
    head = (_normal(seed, 6, (vocab, d)) * 0.02).to(torch.bfloat16).to(torch.float32)
    norm = torch.from_numpy(_norm_weights(seed, 99, d)[0]).to(DEV)
    return table, head, norm, int(np.random.default_rng([int(seed), 9]).integers(vocab))


def _prepare_model(case, seed):
    ctx = qa.GpuContext(0)
    vocab, d = case["vocab"], GEOMETRY[case["geometry"]][0]
    blocks = [_make_block(ctx, seed, i, case, 1, case["context"] + 1) for i in range(case["blocks"])]
    for i, b in enumerate(blocks):
        _fill(b, seed, i, case, [case["context"]])
    table, rows, norm, token = _model_tables(seed, case)
    head = qa.LmHead.from_rows_dev(ctx, rows, vocab, d)
    state = dict(case, ctx=ctx, blocks=blocks, table=table, head=head, norm=norm, token=token, d=d,
                 h=torch.empty(d, dtype=torch.float32, device=DEV),
                 hn=torch.empty(d, dtype=torch.float32, device=DEV),
                 logits=torch.empty(vocab, dtype=torch.float32, device=DEV), stream=torch.cuda.current_stream())
    _run_model(state)
    return state


def _run_model(s):
    embed(s["ctx"], s["table"], s["vocab"], s["d"], [s["token"]], s["h"], s["stream"])
    for block in s["blocks"]:
        if "state_ready" in s:
            block.set_positions([s["context"]])
        block.decode_dev(s["h"], s["context"], s["stream"])
    s["state_ready"] = True
    rms_norm_dev(s["ctx"], s["h"], 1, s["d"], s["norm"], EPS, s["hn"], s["stream"])
    s["head"].logits_dev(s["hn"], 1, s["logits"], s["stream"])
    return [s["logits"], s["h"]]


_PREPARE = {"linear": _prepare_linear, "set": _prepare_set, "sage_blk": _prepare_sage_blk,
            "sage_ref": _prepare_sage_ref, "sage_step": _prepare_sage_step, "exact": _prepare_exact,
            "decode": _prepare_decode, "prefill": _prepare_prefill, "model": _prepare_model}
_RUN = {"linear": _run_linear, "set": _run_set, "sage_blk": _run_sage_blk, "sage_ref": _run_sage_ref,
        "sage_step": _run_sage_step, "exact": _run_exact, "decode": _run_decode, "prefill": _run_prefill,
        "model": _run_model}


# ---- what a pass cannot do without -------------------------------------------

def _layer_work(m, n, r, batch, x_bytes, y_bytes):
    return ((m * r + n * r) / 8 + 2 * (m + n) + batch * (n * x_bytes + m * y_bytes), 2.0 * batch * r * (m + n))


def _pairs(sq, skv, causal):
    return sum(min(skv, max(0, i + skv - sq + 1)) for i in range(sq)) if causal else sq * skv


def _block_work(geometry, rows, pairs, cached_rows, f32=False):
    """Projections over `rows` tokens, attention over `pairs` (query, key) pairs a head, cached rows read once."""
    d, H, Hk, hd, _ = GEOMETRY[geometry]
    bytes_, flops = 2 * rows * d * 4 + 2 * (cached_rows + rows) * Hk * hd * 4, 4.0 * H * hd * pairs
    for m, n in _block_shapes(geometry):
        b, f = _layer_work(m, n, _rank(m, n), 0, 0, 0)
        bytes_, flops = bytes_ + b, flops + 2.0 * rows * _rank(m, n) * (m + n)
    return bytes_, flops


def work(case):
    kind = case["kind"]
    if kind == "linear":
        b, f = _layer_work(case["m"], case["n"], case["r"], case["batch"], 2, 2 if case["y"] == "bfloat16" else 4)
    elif kind == "set":
        each = [_layer_work(m, n, _rank(m, n), case["batch"], 2, 2) for m, n in _block_shapes(case["geometry"])]
        b, f = (case["blocks"] * sum(e[i] for e in each) for i in (0, 1))
    elif kind in ("sage_blk", "sage_ref", "exact"):
        sq, skv = (case["seq_q"], case["seq_kv"]) if kind == "exact" else (case["seq"], case["seq"])
        d, size = (128, 2) if kind == "sage_blk" else (case["d"], 4)
        b = case["batch"] * (2 * case["heads"] * sq + 2 * case["kv_heads"] * skv) * d * size
        f = 4.0 * case["batch"] * case["heads"] * d * _pairs(sq, skv, case["causal"])
    elif kind == "sage_step":
        # the kept codes (one byte a channel) of every cached row, the new block's rows, the query and the result
        b = 2 * case["seq"] * case["kv_heads"] * case["d"] + 8 * case["heads"] * case["d"]
        f = 4.0 * case["seq"] * case["heads"] * case["d"]
    elif kind == "decode":
        c = _contexts(case)
        b, f = _block_work(case["geometry"], len(c), sum(c) + len(c), sum(c) / (4 if case["face"] == "sage" else 1))
    elif kind == "prefill":
        n = case["tokens"]
        b, f = _block_work(case["geometry"], n, n * (n + 1) // 2, 0)
    else:
        c, d = case["context"], GEOMETRY[case["geometry"]][0]
        b, f = _block_work(case["geometry"], 1, c + 1, c / 4)
        b, f = case["blocks"] * b + case["vocab"] * (2 * d + 4), case["blocks"] * f + 2.0 * case["vocab"] * d
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("linear", "set"):  # x scaled, t and u rounded to bf16 on the way
        return {"rel": 1e-2}
    if kind == "sage_blk":         # probabilities and values in fp16, the result in bf16
        return {"rel": 7e-3}
    if kind in ("sage_ref", "sage_step"):  # f32 sums around INT8 codes; a code at a tie may fall either way
        return {"rel": 2e-3}
    if kind == "exact":            # f32 throughout
        return {"rel": 5e-6}
    if kind == "decode" and case["serving"] == "fp32":  # the same; the sage face's codes as above, in one term
        return {"rel": 5e-6 if case["face"] == "exact" else 5e-4}
    return {"rel": 2e-2}           # bf16 at each projection and norm


# ---- the same in 64 bits -----------------------------------------------------

def _signs(packed, n_bits):
    p = torch.from_numpy(packed.copy()).to(DEV)
    bits = (p[:, :, None] >> torch.arange(8, device=DEV, dtype=torch.uint8)) & 1
    return bits.reshape(p.shape[0], -1)[:, :n_bits].to(torch.float64) * 2 - 1


def _linear64(parts, x):
    m, n, r, ub, vt, s1, s2, b = parts
    s1, s2 = (torch.from_numpy(a).to(DEV).double() for a in (s1, s2))
    y = ((x * s2) @ _signs(vt, n).T) @ _signs(ub, r).T * s1
    return y if b is None else y + torch.from_numpy(b).to(DEV).double()


def _attention64(q, k, v, causal):
    """q [..., sq, d] against k, v [..., skv, d] of the same heads, bottom-right causal, 512 queries at a time."""
    sq, skv = q.shape[-2], k.shape[-2]
    out, kt, j = [], k.transpose(-1, -2).contiguous(), torch.arange(skv, device=DEV)
    for i0 in range(0, sq, 512):
        s = torch.matmul(q[..., i0:i0 + 512, :], kt) / math.sqrt(q.shape[-1])
        if causal:
            i = torch.arange(i0, i0 + s.shape[-2], device=DEV)
            s = s.masked_fill(j[None, :] + sq > i[:, None] + skv, -math.inf)
        out.append(torch.matmul(torch.softmax(s, -1), v))
    return torch.cat(out, -2)


def _codes(x, peak):
    scale = torch.where(peak > 0, peak / 127, torch.ones_like(peak))
    return torch.clamp(torch.round(x / scale), -127, 127) * scale


def _block_peak(x, block):
    """The largest magnitude of each run of `block` tokens, over the channels too, spread back over its tokens."""
    s = x.shape[-2]
    peaks = [x[..., a:a + block, :].abs().amax((-1, -2), keepdim=True).expand(*x.shape[:-2], min(block, s - a), 1)
             for a in range(0, s, block)]
    return torch.cat(peaks, -2)


def _sage_blk64(q, k, v, causal):
    """The block-scaled scheme: INT8 q and mean-free k with a scale per 64 tokens, the rest unquantised."""
    q, k = q / math.sqrt(q.shape[-1]), k - k.mean(-2, keepdim=True)
    q, k = _codes(q, _block_peak(q, 64)), _codes(k, _block_peak(k, 64))
    return _attention64(q * math.sqrt(q.shape[-1]), k, v, causal)


def _sage_ref64(q, k, v, causal, block):
    """The reference scheme: per-token q and k codes around each key block's mean, probabilities as INT8 codes
    at 1/127 under the running maximum, values as per-channel codes of the block."""
    s, d = q.shape[-2], q.shape[-1]
    q = _codes(q / math.sqrt(d), (q / math.sqrt(d)).abs().amax(-1, keepdim=True))
    m = torch.full(q.shape[:-1] + (1,), -3e38, dtype=torch.float64, device=DEV)
    total, out = torch.zeros_like(m), torch.zeros_like(q)
    i = torch.arange(s, device=DEV)[:, None]
    for a in range(0, k.shape[-2], block):
        kb, vb = k[..., a:a + block, :], v[..., a:a + block, :]
        mean = kb.mean(-2, keepdim=True)
        kc = _codes(kb - mean, (kb - mean).abs().amax(-1, keepdim=True))
        vc = _codes(vb, vb.abs().amax(-2, keepdim=True))
        sc = torch.matmul(q, (kc + mean).transpose(-1, -2).contiguous())
        if causal:
            sc = sc.masked_fill(a + torch.arange(kb.shape[-2], device=DEV)[None, :] > i, -3e38)
        new = torch.maximum(m, sc.amax(-1, keepdim=True))
        alpha, p = torch.exp(m - new), torch.exp(sc - new)
        if causal:
            p = p.masked_fill(sc < -1e38, 0.0)
        total = alpha * total + p.sum(-1, keepdim=True)
        out = alpha * out + torch.matmul(torch.round(p * 127) / 127, vc)
        m = new
    return out / total


def _heads(x, heads):
    """Rows [t][heads d] to [heads][t][d]."""
    return x.reshape(x.shape[0], heads, -1).transpose(0, 1).contiguous()


def _norm64(h, w):
    return h * torch.rsqrt((h * h).mean(-1, keepdim=True) + EPS) * torch.from_numpy(w).to(DEV).double()


def _rope64(x, positions):
    """x [t][heads][hd], pairs (i, i + hd / 2)."""
    half = x.shape[-1] // 2
    angle = positions.double()[:, None] * THETA ** (-torch.arange(half, device=DEV).double() / half)[None]
    c, s = torch.cos(angle)[:, None], torch.sin(angle)[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _block64(parts, norms, geometry, h, positions, attend):
    """One decoder block over rows h at `positions`; attend(q, k, v) gives the heads' rows."""
    _, H, Hk, hd, _ = GEOMETRY[geometry]
    x, t = _norm64(h, norms[0]), h.shape[0]
    q = _rope64(_linear64(parts[0], x).reshape(t, H, hd), positions)
    k = _rope64(_linear64(parts[1], x).reshape(t, Hk, hd), positions).reshape(t, Hk * hd)
    v = _linear64(parts[2], x)
    h1 = h + _linear64(parts[3], attend(q, k, v).reshape(t, H * hd))
    x = _norm64(h1, norms[1])
    g, u = _linear64(parts[4], x), _linear64(parts[5], x)
    return h1 + _linear64(parts[6], g * u / (1 + torch.exp(-g))), k, v


def _decode64(case, seed, index, h, contexts):
    geometry = case["geometry"]
    d, H, Hk, hd, _ = GEOMETRY[geometry]
    kc, vc = (c.double() for c in _cached_rows(seed, index, len(contexts), max(contexts), Hk * hd))

    def attend(q, k, v):
        rows = []
        for i, c in enumerate(contexts):
            kk, vv = (_heads(torch.cat([x[i, :c], y[i:i + 1]]), Hk).repeat_interleave(H // Hk, 0)
                      for x, y in ((kc, k), (vc, v)))
            qq = q[i][:, None]
            if case.get("face", "sage") == "exact":
                rows.append(_attention64(qq, kk, vv, False)[:, 0])
            else:
                rows.append(_sage_ref64(qq, kk, vv, False, 64)[:, 0])
        return torch.stack(rows)

    return _block64(_block_parts(seed, index, geometry), _norm_weights(seed, index, d), geometry, h,
                    torch.tensor(contexts, device=DEV), attend)


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        return _linear64(_parts(seed, 1, case["m"], case["n"], case["r"], case["bias"]),
                         _linear_x(case, seed).double())
    if kind == "set":
        parts = [p for b in range(case["blocks"]) for p in _block_parts(seed, b, case["geometry"])]
        n, at, out = case["batch"], 0, []
        x = _normal(seed, 3, (n * sum(p[1] for p in parts),)).to(torch.bfloat16).double()
        for p in parts:
            out.append(_linear64(p, x[at:at + n * p[1]].reshape(n, p[1])).reshape(-1))
            at += n * p[1]
        return torch.cat(out)
    if kind in ("sage_blk", "sage_ref", "exact"):
        sq, skv = (case["seq_q"], case["seq_kv"]) if kind == "exact" else (case["seq"], case["seq"])
        d, dtype = (128, torch.bfloat16) if kind == "sage_blk" else (case["d"], torch.float32)
        q, k, v = _attention_inputs(seed, case["batch"], case["heads"], case["kv_heads"], sq, skv, d, dtype)
        group = case["heads"] // case["kv_heads"]
        q, k, v = q.double(), k.double().repeat_interleave(group, 1), v.double().repeat_interleave(group, 1)
        if kind == "sage_blk":
            return _sage_blk64(q, k, v, case["causal"])
        if kind == "sage_ref":
            return _sage_ref64(q, k, v, case["causal"], case["block"])
        return _attention64(q, k, v, case["causal"])
    if kind == "sage_step":
        q, k, v = (x.double() for x in _step_inputs(case, seed))
        group = case["heads"] // case["kv_heads"]
        k, v = (x.transpose(0, 1).repeat_interleave(group, 0).contiguous() for x in (k, v))
        return _sage_ref64(q[:, None], k, v, False, case["block"])[:, 0]
    d = GEOMETRY[case["geometry"]][0]
    if kind == "decode":
        contexts = _contexts(case)
        return list(_decode64(case, seed, 0, _normal(seed, 3, (len(contexts), d)).double(), contexts))
    if kind == "prefill":
        _, H, Hk, _, _ = GEOMETRY[case["geometry"]]
        n = case["tokens"]

        def attend(q, k, v):
            kk, vv = (_heads(x, Hk).repeat_interleave(H // Hk, 0) for x in (k, v))
            return _sage_blk64(q.transpose(0, 1).contiguous(), kk, vv, True).transpose(0, 1)

        h, k, v = _block64(_block_parts(seed, 0, case["geometry"]), _norm_weights(seed, 0, d), case["geometry"],
                           _normal(seed, 3, (n, d)).double(), torch.arange(n, device=DEV), attend)
        return [h, k[None], v[None]]
    table, head, norm, token = _model_tables(seed, case)
    h = table[token][None].double()
    for i in range(case["blocks"]):
        h = _decode64(case, seed, i, h, [case["context"]])[0]
    logits = torch.cat([_norm64(h, norm.cpu().numpy())[0] @ rows.double().T for rows in head.split(16384)])
    return [logits, h[0]]
