"""Performance cases of the KV-cache path: what a serving program has it do.

A case is one layer's share of a pass through the public entry points
(`PagedKvCache`, `RopeTable`, `flash_attention`). Kinds:

  step     a decode step: [window: evict the freed blocks,] append one token
           per sequence, [window: keep the device block table in step,] pick
           the partition for the batch's lengths and attend;
  decode   the attention of a decode step over a cache that is already filled
           (the quantised formats, whose pools are too large to hand back);
  prefill  append a chunk of prompt tokens per sequence, then the chunk's
           causal attention over everything the sequence holds;
  rope     a chunk of projections rotated and appended (it_kv_append_rope);
  append   a chunk of float32 rows quantised and appended;
  export   the cached rows of a batch gathered into contiguous buffers (to
           move a sequence off the device, or to another one);
  op       the Backend FlashAttention operator over contiguous K/V.

Sequence lengths belong to the case (`lens` seeds them); the values, the block
tables and the order of the pool's blocks come from the seed of `prepare`.
Values are N(0, 1), the quantised formats' with 1% of elements 8 times that,
as in the repository's benchmark.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

import infer_train_amd as it
from infer_train_amd.kv import PagedKvCache, RopeTable, flash_attention

_IDS = {"f32": it.F32, "f16": it.F16, "bf16": it.BF16, "q8_0": it.Q8_0, "q4_0": it.Q4_0, "q4_1": it.Q4_1,
        "q5_0": it.Q5_0, "q5_1": it.Q5_1}
_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_BITS = {"f32": 32.0, "f16": 16.0, "bf16": 16.0, "q8_0": 8.5, "q4_0": 4.5, "q4_1": 5.0, "q5_0": 5.5, "q5_1": 6.0}
_QUANT = ("q8_0", "q4_0", "q4_1", "q5_0", "q5_1")
_DEV = "cuda:0"


def listed():
    return [
        # One sequence of 1024 tokens, 12 query heads over 2 KV heads, float32: a single user's next
        # token, where launches and latency are all there is.
        {"name": "step_single_f32", "kind": "step", "dtype": "f32", "heads": 12, "kv_heads": 2, "dim": 128,
         "block": 16, "batch": 1, "lo": 1024, "hi": 1024, "window": 0, "lens": 1},
        # A mixed batch: 32 sequences of 256 to 4096 tokens.
        {"name": "step_ragged_bf16", "kind": "step", "dtype": "bf16", "heads": 28, "kv_heads": 4, "dim": 128,
         "block": 16, "batch": 32, "lo": 256, "hi": 4096, "window": 0, "lens": 2},
        # Sliding windows: 64 sequences far into their text, each reading its last 4096 positions.
        {"name": "step_window_bf16", "kind": "step", "dtype": "bf16", "heads": 16, "kv_heads": 2, "dim": 128,
         "block": 16, "batch": 64, "lo": 30000, "hi": 32768, "window": 4096, "lens": 4},
        # Long contexts with a compressed cache: the largest decode.
        {"name": "decode_long_q8_0", "kind": "decode", "dtype": "q8_0", "heads": 24, "kv_heads": 4, "dim": 256,
         "block": 32, "batch": 16, "lo": 32768, "hi": 131072, "lens": 5},
        # A 4-bit cache at middle lengths.
        {"name": "decode_q4_0", "kind": "decode", "dtype": "q4_0", "heads": 32, "kv_heads": 8, "dim": 128,
         "block": 16, "batch": 16, "lo": 2048, "hi": 16384, "lens": 6},
        # Chunked prefill in a batch: 8 sequences of 2048 cached tokens each take a 512-token chunk.
        {"name": "prefill_chunk_bf16", "kind": "prefill", "dtype": "bf16", "heads": 32, "kv_heads": 8, "dim": 128,
         "block": 16, "batch": 8, "lo": 2048, "hi": 2048, "chunk_lo": 512, "chunk_hi": 512, "causal": True, "lens": 3},
        # New prompts of any length with nothing cached yet.
        {"name": "prefill_prompts_f16", "kind": "prefill", "dtype": "f16", "heads": 28, "kv_heads": 4, "dim": 128,
         "block": 16, "batch": 6, "lo": 0, "hi": 0, "chunk_lo": 65, "chunk_hi": 1500, "causal": True, "lens": 7},
        # One user's long document, fed in chunks: few query rows, many keys.
        {"name": "prefill_long_bf16", "kind": "prefill", "dtype": "bf16", "heads": 32, "kv_heads": 8, "dim": 128,
         "block": 16, "batch": 1, "lo": 16000, "hi": 16000, "chunk_lo": 500, "chunk_hi": 500, "causal": True, "lens": 8},
        # The projections of that chunked prefill before its attention: rotate and store.
        {"name": "rope_chunk_bf16", "kind": "rope", "dtype": "bf16", "heads": 32, "kv_heads": 8, "dim": 128,
         "block": 16, "batch": 8, "lo": 2048, "hi": 2048, "chunk_lo": 512, "chunk_hi": 512, "lens": 3},
        # The same chunk stored in a 4-bit cache.
        {"name": "append_chunk_q4_0", "kind": "append", "dtype": "q4_0", "heads": 24, "kv_heads": 4, "dim": 256,
         "block": 32, "batch": 8, "lo": 2048, "hi": 2048, "chunk_lo": 512, "chunk_hi": 512, "lens": 3},
        # Compressed rows of a few sequences, packed records for another device.
        {"name": "export_q8_0", "kind": "export", "dtype": "q8_0", "heads": 24, "kv_heads": 4, "dim": 256,
         "block": 32, "batch": 4, "lo": 4096, "hi": 16384, "lens": 9},
        # The operator as the reference's backend offers it, with its additive mask.
        {"name": "op_flash_f32", "kind": "op", "heads": 12, "dim": 128, "n_kv": 2000, "mask": True, "lens": 10},
    ]


# (query heads, KV heads, head dim) of the repository's configurations and tests.
_HEADS = ((12, 2, 128), (28, 4, 128), (32, 8, 128), (16, 2, 128), (24, 4, 256), (8, 8, 128), (10, 2, 128), (6, 2, 256),
          (16, 8, 256), (9, 3, 128))


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choice(("step", "step", "step", "decode", "decode", "prefill", "prefill", "prefill", "rope", "append",
                       "export", "op"))
    heads, kv, dim = rng.choice(_HEADS)
    c = {"kind": kind, "heads": heads, "dim": dim, "lens": rng.randrange(1 << 20)}
    if kind == "op":
        return dict(c, n_kv=_log(rng, 1, 16384), mask=rng.random() < 0.5)
    c.update(kv_heads=kv, block=rng.choice((8, 16, 16, 32, 64)))
    if kind == "step":
        c["dtype"] = rng.choice(("bf16", "bf16", "f16", "f32"))
        c["batch"] = _log(rng, 1, 96)
        c["hi"] = _log(rng, 16, 32768)
        c["lo"] = rng.choice((c["hi"], max(1, c["hi"] // 16), max(1, c["hi"] // 2)))
        c["window"] = rng.choice((0, 0, 512, 1000, 4096))
    elif kind in ("decode", "export"):
        c["dtype"] = rng.choice(_QUANT if kind == "decode" else _QUANT + ("bf16", "f16", "f32"))
        c["batch"] = _log(rng, 1, 48)
        c["hi"] = _log(rng, 64, 131072 if kind == "decode" else 16384)
        c["lo"] = rng.choice((c["hi"], max(1, c["hi"] // 8), max(1, c["hi"] // 2)))
    else:
        if kind == "prefill":
            c["dtype"] = rng.choice(("bf16", "bf16", "f16"))
            c["dim"], c["causal"] = 128, rng.random() < 0.85
        else:
            c["dtype"] = rng.choice(_QUANT if kind == "append" else ("bf16", "bf16", "f16", "f32") + _QUANT)
        c["batch"] = _log(rng, 1, 24)
        c["hi"] = rng.choice((0, _log(rng, 16, 32768)))
        c["lo"] = rng.choice((c["hi"], c["hi"] // 4))
        c["chunk_hi"] = _log(rng, 1, 4096)
        c["chunk_lo"] = rng.choice((c["chunk_hi"], max(1, c["chunk_hi"] // 8)))
    return c


def draw(rng):
    """A case of the listed ones' ranges that costs no more than the largest of its kind may."""
    while True:
        c = _draw_once(rng)
        w = work(c)
        rows = 0 if c["kind"] == "op" else sum(ctx - st for ctx, _, st in _lengths(c))
        pool = rows * c.get("kv_heads", 1) * c["dim"] * _BITS[c.get("dtype", "f32")] / 4  # bits of K and V
        if c["kind"] == "decode":
            ok = w["bytes"] <= 2.5e9
        else:
            ok = w["bytes"] <= 8e8 and pool <= 8e8
        if ok and w["flops"] <= 1.5e11:
            return c


def _lengths(c):
    """[(tokens after the pass, tokens the pass adds, window start)] of each sequence."""
    r = random.Random(c["lens"])
    out = []
    for _ in range(c["batch"]):
        n = r.randint(c["lo"], c["hi"])
        if c["kind"] == "step":
            out.append((n, 1, max(0, n - c["window"]) if c["window"] else 0))
        elif c["kind"] in ("decode", "export"):
            out.append((n, 0, 0))
        else:
            q = r.randint(c["chunk_lo"], c["chunk_hi"])
            out.append((n + q, q, 0))
    return out


def _keys_attended(c):
    """Query rows x keys over the pass, per query head."""
    total = 0
    for ctx, new, st in _lengths(c):
        if c["kind"] == "prefill":
            total += (new * (ctx - new) + new * (new + 1) // 2) if c["causal"] else new * ctx
        else:
            total += ctx - st
    return total


def work(c):
    if c["kind"] == "op":
        q, kv = c["heads"] * c["dim"] * 4, c["n_kv"] * c["dim"] * 4
        return {"bytes": 2 * q + 2 * kv + (c["n_kv"] * 4 if c["mask"] else 0), "flops": 4 * c["heads"] * c["dim"] * c["n_kv"]}
    lens = _lengths(c)
    row = 2 * c["kv_heads"] * c["dim"] * _BITS[c["dtype"]] / 8  # K and V of one cached token
    new = sum(n for _, n, _ in lens)
    held = sum(ctx - st for ctx, _, st in lens)
    qbytes = {"f16": 2, "bf16": 2}.get(c["dtype"], 4) * c["heads"] * c["dim"]
    src = 2 * c["kv_heads"] * c["dim"] * 4
    if c["kind"] == "step":
        return {"bytes": held * row + 2 * new * row + 2 * len(lens) * qbytes, "flops": 4 * c["dim"] * c["heads"] * held}
    if c["kind"] == "decode":
        return {"bytes": held * row + 2 * len(lens) * qbytes, "flops": 4 * c["dim"] * c["heads"] * held}
    if c["kind"] == "prefill":
        return {"bytes": held * row + 2 * new * row + 2 * new * qbytes, "flops": 4 * c["dim"] * c["heads"] * _keys_attended(c)}
    if c["kind"] == "rope":
        return {"bytes": new * (src + row + c["heads"] * c["dim"] * 4 + qbytes), "flops": 6 * new * c["dim"] * (c["heads"] + c["kv_heads"])}
    if c["kind"] == "append":
        return {"bytes": new * (src + row), "flops": 0}
    return {"bytes": 2 * held * row, "flops": 0}


def tolerance(c):
    """About four times what the path shows against `exact`: the rounding of 16-bit outputs and
    probabilities, or float32 sums. Moved, rotated and quantised bytes are what the CPU computes."""
    if c["kind"] in ("rope", "append", "export"):
        return "exact"
    return {"rel": {"bf16": 1e-2, "f16": 1.5e-3}.get(c.get("dtype"), 4e-6)}


# ---- inputs -----------------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device=_DEV)
    g.manual_seed(seed)
    return g


def _normal(g, *shape, outliers=False):
    x = torch.randn(shape, generator=g, device=_DEV)
    if outliers:
        x = torch.where(torch.rand(shape, generator=g, device=_DEV) < 0.01, 8 * x, x)
    return x


def _page_bytes(c):
    return int(c["block"] * c["dim"] * _BITS[c["dtype"]] / 8)


def _quantise(x, fmt):
    """Page bytes [..., page] of rows x [..., block, dim] in a quantised format's page layout."""
    bs, dim = x.shape[-2:]
    lead, ng = x.shape[:-2], dim // 32
    g = x.reshape(*lead, bs, ng, 32)

    def bytes_of(t, dt):
        return t.to(dt).contiguous().view(torch.uint8).reshape(*lead, bs, -1)

    if fmt == "q8_0":
        d = g.abs().amax(-1, keepdim=True) / 127
        q = torch.round(g / torch.where(d > 0, d, 1.0))
        return torch.cat([bytes_of(q, torch.int8).reshape(*lead, -1), bytes_of(d, torch.float16).reshape(*lead, -1)], -1)
    top = 15 if fmt[1] == "4" else 31
    half = (top + 1) // 2
    if fmt[3] == "0":
        m = torch.gather(g, -1, g.abs().argmax(-1, keepdim=True))
        d = m / -half
        q = torch.floor(g / torch.where(d != 0, d, 1.0) + (half + 0.5)).clamp(0, top)
        meta = bytes_of(d, torch.float16)
    else:
        lo = g.amin(-1, keepdim=True)
        d = (g.amax(-1, keepdim=True) - lo) / top
        q = torch.floor((g - lo) / torch.where(d != 0, d, 1.0) + 0.5).clamp(0, top)
        meta = bytes_of(torch.cat([d, lo], -1), torch.float16)
    q = q.to(torch.uint8)
    nib = (q[..., :16] & 15) | ((q[..., 16:] & 15) << 4)
    if fmt[1] == "5":
        bit = torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], dtype=torch.uint8, device=x.device)
        qh = ((q >> 4).reshape(*lead, bs, ng, 4, 8) * bit).sum(-1, dtype=torch.uint8)
        meta = torch.cat([qh.reshape(*lead, bs, -1), meta], -1)
    return torch.cat([nib.reshape(*lead, -1), meta.reshape(*lead, -1)], -1)


def _fill(c, g, n_blocks):
    """A pool's bytes as earlier passes left them, as plain torch makes them."""
    kv, bs, dim = c["kv_heads"], c["block"], c["dim"]
    if c["dtype"] in _TORCH:
        return torch.randn((n_blocks, kv, bs, dim), generator=g, device=_DEV).to(_TORCH[c["dtype"]]).view(torch.uint8).reshape(-1)
    pool = torch.empty((n_blocks, kv, _page_bytes(c)), dtype=torch.uint8, device=_DEV)
    step = max(1, (1 << 27) // (kv * bs * dim))
    for b in range(0, n_blocks, step):
        n = min(step, n_blocks - b)
        pool[b:b + n] = _quantise(_normal(g, n, kv, bs, dim, outliers=True), c["dtype"])
    return pool.reshape(-1)


def _inputs(c, seed):
    """Everything `prepare` gives the path, as plain tensors."""
    g = _gen(seed)
    if c["kind"] == "op":
        x = {"q": _normal(g, c["heads"], c["dim"]), "k": _normal(g, c["n_kv"], c["dim"]), "v": _normal(g, c["n_kv"], c["dim"])}
        if c["mask"]:
            m = 0.5 * _normal(g, c["n_kv"])
            hidden = torch.rand(c["n_kv"], generator=g, device=_DEV) < 0.1
            hidden[0] = False  # at least one key is seen
            x["mask"] = torch.where(hidden, -math.inf, m)
        return x
    lens, bs, kv, dim = _lengths(c), c["block"], c["kv_heads"], c["dim"]
    held = [(st // bs, (ctx - 1) // bs + 1) for ctx, _, st in lens]
    spare = max(1, len(lens) // bs)  # blocks the window gave back
    n_blocks = sum(b - a for a, b in held) + spare
    order = np.random.RandomState(seed % (1 << 32)).permutation(n_blocks).astype(np.int32)
    tables = np.full((len(lens), max(b for _, b in held)), -1, np.int32)
    at = 0
    for i, (a, b) in enumerate(held):
        tables[i, a:b] = order[at:at + b - a]
        at += b - a
    seq = np.repeat(np.arange(len(lens), dtype=np.int32), [n for _, n, _ in lens])
    pos = np.concatenate([np.arange(ctx - n, ctx, dtype=np.int32) for ctx, n, _ in lens])
    slots = tables[seq, pos // bs].astype(np.int64) * bs + pos % bs
    on = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(_DEV)  # noqa: E731
    ctx = np.array([n for n, _, _ in lens], np.int32)
    start = np.array([s for _, _, s in lens], np.int32)
    x = {"n_blocks": n_blocks, "tables": on(tables), "ctx": on(ctx), "ctx_host": ctx, "start_host": start,
         "start": on(start) if c.get("window") else None, "seq": on(seq), "pos": on(pos), "slots": on(slots),
         "freed": on(order[at:]), "longest": int((ctx - start).max())}
    x["k_pool"], x["v_pool"] = _fill(c, g, n_blocks), _fill(c, g, n_blocks)
    n = len(seq)
    src = torch.float32 if c["kind"] in ("rope", "append") else _TORCH.get(c["dtype"], torch.float32)
    if n:
        x["k"], x["v"] = (_normal(g, n, kv, dim, outliers=c["dtype"] in _QUANT).to(src) for _ in range(2))
    if c["kind"] in ("step", "decode", "prefill", "rope"):
        rows = n if c["kind"] in ("prefill", "rope") else len(lens)
        x["q"] = _normal(g, rows, c["heads"], dim).to(src)
    if c["kind"] == "prefill":
        x["cu_q"] = on(np.concatenate([[0], np.cumsum([m for _, m, _ in lens])]).astype(np.int32))
        x["longest_q"] = max(m for _, m, _ in lens)
    if c["kind"] == "export":
        x["cu_out"] = on(np.concatenate([[0], np.cumsum(ctx)[:-1]]).astype(np.int64))
        x["out_bytes"] = int(ctx.sum()) * kv * _page_bytes(c) // bs
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    x["case"] = case
    if case["kind"] == "op":
        return x
    cache = PagedKvCache(x["n_blocks"], case["block"], case["kv_heads"], case["dim"], _IDS[case["dtype"]])
    cache.k_pool.copy_(x.pop("k_pool"))
    cache.v_pool.copy_(x.pop("v_pool"))
    x["cache"] = cache
    if case["kind"] == "rope":
        x["rope"] = RopeTable(case["dim"], int(x["ctx_host"].max()), 10000.0)
    if case["kind"] == "export":
        x["k_out"], x["v_out"] = (torch.empty(x["out_bytes"], dtype=torch.uint8, device=_DEV) for _ in range(2))
    return x


# ---- one pass ---------------------------------------------------------------------------------


def _pools(case, cache):
    if case["dtype"] in _TORCH:
        return [cache.view("k"), cache.view("v")]
    return [cache.k_pool, cache.v_pool]


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "op":
        return flash_attention(s["q"], s["k"], s["v"], s.get("mask"))
    cache = s["cache"]
    if kind in ("step", "decode"):
        if kind == "step":
            if case["window"]:
                cache.evict(s["freed"])
            cache.append(s["k"], s["v"], s["slots"])
            if case["window"]:
                cache.sync_tables(s["tables"], s["seq"], s["pos"], s["slots"])
        part = cache.decode_partition(case["heads"], s["ctx_host"], s["start_host"])
        out = cache.decode(s["q"], s["tables"], s["ctx"], s["start"], s["longest"], partition=part)
        return out if kind == "decode" else [out, s["tables"]] + _pools(case, cache)
    if kind == "prefill":
        cache.append(s["k"], s["v"], s["slots"])
        out = cache.prefill(s["q"], s["cu_q"], s["longest_q"], s["tables"], s["ctx"], causal=case["causal"])
        return [out] + _pools(case, cache)
    if kind == "rope":
        q_type = _TORCH[case["dtype"]] if case["dtype"] in _TORCH else torch.float32
        q = cache.append_rope(s["rope"], s["q"], s["k"], s["v"], s["slots"], s["pos"], q_out_dtype=q_type)
        return [q] + _pools(case, cache)
    if kind == "append":
        cache.append(s["k"], s["v"], s["slots"])
        return _pools(case, cache)
    cache.gather(s["tables"], s["ctx"], None, s["cu_out"], s["longest"], s["k_out"], s["v_out"])
    return [s["k_out"], s["v_out"]]


# ---- the same in 64 bits ----------------------------------------------------------------------


def _rows64(c, pool, blocks):
    """float64 rows [kv_heads, tokens, dim] of a list of blocks of a pool's bytes."""
    kv, bs, dim = c["kv_heads"], c["block"], c["dim"]
    pages = pool.view(-1, kv, _page_bytes(c))[blocks.long()]
    n, fmt = pages.shape[0], c["dtype"]
    if fmt in _TORCH:
        x = pages.contiguous().view(_TORCH[fmt]).double()
    else:
        ng = dim // 32
        f16 = lambda b, k: b.contiguous().view(torch.float16).double().reshape(n, kv, bs, ng, k)  # noqa: E731
        main = bs * dim if fmt == "q8_0" else bs * dim // 2
        qs, side = pages[..., :main].contiguous(), pages[..., main:].reshape(n, kv, bs, -1)
        if fmt == "q8_0":
            x = qs.view(torch.int8).double().reshape(n, kv, bs, ng, 32) * f16(side, 1)
        else:
            nib = qs.reshape(n, kv, bs, ng, 16)
            q = torch.cat([nib & 15, nib >> 4], -1).double()
            if fmt[1] == "5":
                qh = side[..., :4 * ng].reshape(n, kv, bs, ng, 4, 1)
                shift = torch.arange(8, device=pool.device, dtype=torch.uint8)
                q = q + 16 * ((qh >> shift) & 1).reshape(n, kv, bs, ng, 32).double()
                side = side[..., 4 * ng:]
            if fmt[3] == "0":
                x = f16(side, 1) * (q - (8 if fmt[1] == "4" else 16))
            else:
                dm = f16(side, 2)
                x = dm[..., :1] * q + dm[..., 1:]
    return x.reshape(n, kv, bs, dim).transpose(0, 1).reshape(kv, n * bs, dim)


def exact(case, seed):
    if case["kind"] in ("append", "export"):
        return None
    x = _inputs(case, seed)
    if case["kind"] == "op":
        s = x["q"].double() @ x["k"].double().t().contiguous() / math.sqrt(case["dim"])
        if case["mask"]:
            s = s + x["mask"].double()
        return torch.softmax(s, -1) @ x["v"].double()
    heads, kv, dim, bs = case["heads"], case["kv_heads"], case["dim"], case["block"]
    if case["kind"] == "rope":
        p = torch.arange(dim // 2, device=_DEV, dtype=torch.float32)
        theta = (x["pos"].float()[:, None] * torch.pow(10000.0, -2 * p / dim)).double()[:, None]
        a, b = x["q"][..., 0::2].double(), x["q"][..., 1::2].double()
        cos, sin = torch.cos(theta), torch.sin(theta)
        return [torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(x["q"].shape), None, None]
    out = torch.empty(x["q"].shape, dtype=torch.float64, device=_DEV)
    at = 0
    for i, (ctx, new, st) in enumerate(_lengths(case)):
        first = st // bs
        blocks = x["tables"][i, first:(ctx - 1) // bs + 1]
        q0, rows = (at, new) if case["kind"] == "prefill" else (i, 1)
        k, v = (_rows64(case, x[p], blocks) for p in ("k_pool", "v_pool"))
        if new:
            k[:, ctx - new - first * bs:ctx - first * bs] = x["k"][at:at + new].double().transpose(0, 1)
            v[:, ctx - new - first * bs:ctx - first * bs] = x["v"][at:at + new].double().transpose(0, 1)
        k, v = k[:, st - first * bs:ctx - first * bs], v[:, st - first * bs:ctx - first * bs]
        for h in range(kv):
            group = slice(h * (heads // kv), (h + 1) * (heads // kv))
            kt, vh = k[h].t().contiguous(), v[h].contiguous()
            for r in range(0, rows, 512):
                n = min(512, rows - r)
                q = x["q"][q0 + r:q0 + r + n, group].double()
                s = (q.reshape(-1, dim) @ kt / math.sqrt(dim)).reshape(n, -1, ctx - st)
                if case["kind"] == "prefill" and case["causal"]:
                    key, query = torch.arange(ctx, device=_DEV), torch.arange(ctx - new + r, ctx - new + r + n, device=_DEV)
                    s = s.masked_fill(key[None, None, :] > query[:, None, None], -math.inf)
                out[q0 + r:q0 + r + n, group] = (torch.softmax(s, -1).reshape(-1, ctx - st) @ vh).reshape(n, -1, dim)
        at += new
    if case["kind"] == "decode":
        return out
    return [out] + [None] * (3 if case["kind"] == "step" else 2)
