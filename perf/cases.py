"""The work a program has this package do, as cases to time.

Four kinds, each through public entry points:

* ``paged``    one decode step over the paged KV cache: ``PagedDecode`` (prepared once, as a
               serving loop holds it), with ``kv_append`` of the step's token where ``append``;
* ``sdpa``     one ``scaled_dot_product_attention`` call with dense K / V: prompts, chunks of
               prompts against a cache, encoders, decode steps, with the masks these come with;
* ``relayout`` a tensor moved host order -> sticks -> (transposed sticks) -> host order by
               prepared ``DmaCopy``s, as weights and activations are;
* ``pages``    a prompt's dense K / V turned into cache pages (``dense_to_pages``), the step
               between prefill and paged decode.

A case holds sizes only; contexts and padded lengths of a batch follow from them by a fixed
low-discrepancy sequence, so that ``work`` needs no seed.
"""

from __future__ import annotations

import math

import torch

PAGE = 64
GOLDEN = 0.6180339887498949
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
# (q heads, KV heads, head_dim) of this repository's benchmark and tests.
HEADS = [(32, 8, 128), (64, 8, 128), (16, 16, 64), (32, 32, 128), (8, 8, 64)]


def _paged(name, batch, heads, ctx_min, ctx_max, append):
    c = {"kind": "paged", "batch": batch, "q_heads": heads[0], "kv_heads": heads[1], "head_dim": heads[2],
         "ctx_min": ctx_min, "ctx_max": ctx_max, "append": append}
    return {"name": name, **c} if name else c


def _sdpa(name, batch, heads, q_len, kv_len, mask, lse=False):
    c = {"kind": "sdpa", "batch": batch, "q_heads": heads[0], "kv_heads": heads[1], "head_dim": heads[2],
         "q_len": q_len, "kv_len": kv_len, "mask": mask, "lse": lse}
    return {"name": name, **c} if name else c


def _relayout(name, lead, rows, cols, dtype, restick):
    c = {"kind": "relayout", "lead": lead, "rows": rows, "cols": cols, "dtype": dtype, "restick": restick}
    return {"name": name, **c} if name else c


def _pages(name, batch, kv_heads, head_dim, length):
    c = {"kind": "pages", "batch": batch, "kv_heads": kv_heads, "head_dim": head_dim, "length": length}
    return {"name": name, **c} if name else c


def listed():
    return [
        # One user, a short chat so far: append the token, attend.  Latency and launches.
        _paged("paged_one", 1, (32, 8, 128), 700, 700, True),
        # The benchmark's step: 32 sequences of 4096 tokens, 32 / 8 heads.
        _paged("paged_batch", 32, (32, 8, 128), 4096, 4096, False),
        # Continuous batching: 64 sequences anywhere between 128 and 32768 tokens (the benchmark's
        # ragged batch, and the largest call here).
        _paged("paged_ragged", 64, (32, 8, 128), 128, 32768, False),
        # A decode step of a padded batch over a static dense cache: a boolean key mask [B, 1, 1, S]
        # tells each sequence's real keys.
        _sdpa("decode_padded", 16, (32, 8, 128), 1, 2048, "pad"),
        # An ordinary prompt of no particular length, causal.
        _sdpa("prompt", 1, (32, 8, 128), 1000, 1000, "causal"),
        # The benchmark's long prompt, causal.
        _sdpa("prompt_long", 1, (32, 8, 128), 4096, 4096, "causal"),
        # An encoder's batch, padded to its longest text; multi-head, head_dim 64.
        _sdpa("encoder_padded", 8, (16, 16, 64), 384, 384, "pad"),
        # Attention with a learned relative-position bias kept in fp32 [1, H, S, S].
        _sdpa("position_bias", 2, (16, 16, 64), 777, 777, "bias_f32"),
        # Chunked prefill: 128 new tokens of 4 sequences against 4096 cached keys, the chunk's own
        # tokens causal (a boolean mask aligned to the last key); the logsumexp joins chunks.
        _sdpa("chunk", 4, (32, 8, 128), 128, 4096, "tail", lse=True),
        # A weight matrix: host order -> sticks, its transpose-restick, and back (the benchmark's
        # three relayouts).
        _relayout("matrix", 1, 4096, 4096, "f16", True),
        # Activations or logits of odd sizes, fp32, to the device layout and back.
        _relayout("activations", 3, 1021, 2500, "f32", False),
        # The KV of 8 finished prompts of 3000 tokens handed to the paged cache.
        _pages("prompt_to_pages", 8, 8, 128, 3000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["paged", "paged", "decode", "decode", "prompt", "prompt", "prompt", "chunk", "chunk",
                       "relayout", "relayout", "pages"])
    if kind == "paged":
        heads = rng.choice(HEADS)
        batch = _log_int(rng, 1, 64)
        hi = _log_int(rng, 64, min(32768, (1 << 30) // (batch * heads[1] * heads[2])))
        lo = hi if rng.random() < 0.3 else max(1, int(hi * rng.uniform(0.02, 0.9)))
        return _paged(None, batch, heads, lo, hi, batch * hi <= 4096)
    if kind == "decode":
        heads = rng.choice(HEADS)
        kv = _log_int(rng, 64, 8192)
        batch = _log_int(rng, 1, max(1, min(64, (1 << 18) // kv)))
        return _sdpa(None, batch, heads, 1, kv, rng.choice(["none", "pad", "pad_f16"]))
    if kind == "prompt":
        heads = rng.choice(HEADS)
        n = _log_int(rng, 48, 4096)
        mask = rng.choice(["causal", "causal", "none", "pad", "causal_f16", "bias_f32"])
        if mask == "bias_f32":
            n = min(n, 2048)
        batch = _log_int(rng, 1, max(1, min(16, (1 << 22) // (n * n))))
        return _sdpa(None, batch, heads, n, n, mask)
    if kind == "chunk":
        heads = rng.choice(HEADS)
        q = _log_int(rng, 8, 512)
        kv = max(q, _log_int(rng, 256, 8192))
        batch = _log_int(rng, 1, max(1, min(8, (1 << 21) // (q * kv))))
        return _sdpa(None, batch, heads, q, kv, rng.choice(["tail", "none"]), lse=True)
    if kind == "relayout":
        lead = rng.choice([1, 1, 2, 3, 8])
        rows, cols = _log_int(rng, 16, 4096), _log_int(rng, 64, 8192)
        dtype = rng.choice(["f16", "f16", "bf16", "f32"])
        restick = lead == 1 and dtype != "f32" and rng.random() < 0.5
        if restick:  # tilings of whole sticks nest
            rows, cols = -(-rows // 64) * 64, -(-cols // 64) * 64
        return _relayout(None, lead, rows, cols, dtype, restick)
    return _pages(None, _log_int(rng, 1, 16), rng.choice([8, 16]), rng.choice([64, 128]), _log_int(rng, 100, 4096))


# ---------------------------------------------------------------- sizes --

def _spread(n, lo, hi):
    """n whole numbers between lo and hi, the first of them hi."""
    return [hi] + [lo + int((hi - lo + 1) * ((i * GOLDEN) % 1.0)) for i in range(1, n)]


def _contexts(case):
    return _spread(case["batch"], case["ctx_min"], case["ctx_max"])


def _lengths(case):
    """Real keys of each sequence of a padded batch."""
    return _spread(case["batch"], max(1, (2 * case["kv_len"]) // 5), case["kv_len"])


def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 64 + what) % (1 << 62))


def _randn(shape, seed, what, dtype=torch.float16):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(generator=_gen(seed, what))


# --------------------------------------------------------------- inputs --

def _paged_inputs(case, seed):
    Hq, Hkv, D = case["q_heads"], case["kv_heads"], case["head_dim"]
    ctx = _contexts(case)
    pages = [-(-c // PAGE) for c in ctx]
    total = sum(pages)
    k = _randn((total, Hkv, D // 64, PAGE, 64), seed, 0)
    v = _randn((total, Hkv, D, PAGE), seed, 1)
    q = _randn((len(ctx), Hq, D), seed, 2)
    k_new = _randn((len(ctx), Hkv, D), seed, 3)
    v_new = _randn((len(ctx), Hkv, D), seed, 4)
    perm = torch.randperm(total, generator=torch.Generator().manual_seed(int(seed) % (1 << 62)), dtype=torch.int64)
    table = torch.zeros((len(ctx), max(pages)), dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = perm[at:at + n].to(torch.int32)
        at += n
    return q, k, v, table.cuda(), ctx, k_new, v_new


def _mask(case, seed):
    B, Hq, Sq, Skv = case["batch"], case["q_heads"], case["q_len"], case["kv_len"]
    kind = case["mask"]
    if kind in ("none", "causal"):
        return None
    if kind in ("pad", "pad_f16", "causal_f16"):
        lens = torch.tensor(_lengths(case), device="cuda")
        keep = (torch.arange(Skv, device="cuda")[None, :] < lens[:, None])[:, None, None, :]
        if kind == "pad":
            return keep
        if kind == "causal_f16":  # a padded batch of prompts, both rules in one additive mask
            keep = keep & torch.ones((Sq, Skv), dtype=torch.bool, device="cuda").tril()
        zero = torch.zeros(keep.shape, dtype=torch.float16, device="cuda")
        return zero.masked_fill_(~keep, torch.finfo(torch.float16).min)
    if kind == "tail":  # query i is key Skv - Sq + i
        return torch.ones((Sq, Skv), dtype=torch.bool, device="cuda").tril(Skv - Sq)[None, None]
    assert kind == "bias_f32"
    table = _randn((Hq, Sq + Skv - 1), seed, 8, torch.float32)  # one value per head and distance
    at = torch.arange(Skv, device="cuda")[None, :] - torch.arange(Sq, device="cuda")[:, None] + Sq - 1
    return table[:, at][None].contiguous()


def _sdpa_inputs(case, seed):
    """q, k, v as a model's projections leave them: [B, S, H, D] viewed as [B, H, S, D] for
    prompts; a decode step's or a chunk's K / V is a cache [B, Hkv, S, D]."""
    B, Hq, Hkv, D = case["batch"], case["q_heads"], case["kv_heads"], case["head_dim"]
    Sq, Skv = case["q_len"], case["kv_len"]
    q = _randn((B, Sq, Hq, D), seed, 5).transpose(1, 2)
    if Sq == Skv:
        k, v = (_randn((B, Skv, Hkv, D), seed, w).transpose(1, 2) for w in (6, 7))
    else:
        k, v = (_randn((B, Hkv, Skv, D), seed, w) for w in (6, 7))
    return q, k, v, _mask(case, seed)


def _host_size(case):
    return [case["rows"], case["cols"]] if case["lead"] == 1 else [case["lead"], case["rows"], case["cols"]]


def prepare(case, seed):
    import torch_spyre_amd as tsa

    if case["kind"] == "paged":
        q, k, v, table, ctx, k_new, v_new = _paged_inputs(case, seed)
        lens = torch.tensor(ctx, dtype=torch.int32, device="cuda")
        lse = torch.empty((len(ctx), case["q_heads"]), dtype=torch.float32, device="cuda")
        call = tsa.PagedDecode(q, k, v, table, lens, max_context_len=max(ctx), lse=lse)
        step = (k_new, v_new, k, v, table, lens - 1) if case["append"] else None
        return {"kind": "paged", "call": call, "append": step, "lse": lse, "keep": (q, lens)}
    if case["kind"] == "sdpa":
        q, k, v, mask = _sdpa_inputs(case, seed)
        kw = {"attn_mask": mask, "is_causal": case["mask"] == "causal", "enable_gqa": case["q_heads"] != case["kv_heads"],
              "return_lse": case["lse"]}
        return {"kind": "sdpa", "qkv": (q, k, v), "kw": kw}
    if case["kind"] == "relayout":
        size, dtype = _host_size(case), DTYPES[case["dtype"]]
        x = _randn(size, seed, 9, dtype)
        stride = list(x.stride())
        layout = tsa.SpyreTensorLayout(size, dtype)
        dev = tsa.spyre_empty_with_layout(size, stride, dtype, layout)
        back = torch.empty_like(x)
        buf = tsa.device_buffer(dev)
        copies = [tsa.DmaCopy(x, buf, tsa.dma_plan(size, stride, stride, 0, layout, True))]
        outs = [buf]
        if case["restick"]:
            other = tsa.transpose_restick_layout(case["rows"], case["cols"], dtype)
            turned = tsa.device_buffer(tsa.spyre_empty_with_layout(size, stride, dtype, other))
            copies.append(tsa.DmaCopy(buf, turned, [tsa.restick_plan(size, layout, other)]))
            outs.append(turned)
        copies.append(tsa.DmaCopy(buf, back, tsa.dma_plan(size, stride, stride, 0, layout, False)))
        return {"kind": "relayout", "copies": copies, "outs": outs + [back], "keep": x}
    shape = (case["batch"], case["kv_heads"], case["length"], case["head_dim"])
    return {"kind": "pages", "kv": (_randn(shape, seed, 10), _randn(shape, seed, 11))}


def run(state):
    import torch_spyre_amd as tsa

    if state["kind"] == "paged":
        if state["append"] is None:
            return state["call"](), state["lse"]
        step = state["append"]
        tsa.kv_append(*step)
        return state["call"](), state["lse"], step[2], step[3]
    if state["kind"] == "sdpa":
        return tsa.scaled_dot_product_attention(*state["qkv"], **state["kw"])
    if state["kind"] == "relayout":
        for copy in state["copies"]:
            copy()
        return state["outs"]
    cache, table = tsa.dense_to_pages(*state["kv"])
    return cache.k, cache.v, table


# ----------------------------------------------------------------- work --

def _pairs(case):
    """(query, key) pairs that a head attends, over the batch."""
    B, Sq, Skv, kind = case["batch"], case["q_len"], case["kv_len"], case["mask"]
    if kind in ("none", "bias_f32"):
        return B * Sq * Skv
    if kind == "causal":  # Sq == Skv in every causal case
        return B * Sq * (Sq + 1) // 2
    if kind == "tail":
        return B * (Sq * (Skv - Sq) + Sq * (Sq + 1) // 2)
    lens = _lengths(case)
    if kind == "causal_f16":
        return sum(n * (n + 1) // 2 + (Sq - n) * n for n in lens)
    return Sq * sum(lens)


def work(case):
    if case["kind"] == "paged":
        ctx, Hq, Hkv, D = _contexts(case), case["q_heads"], case["kv_heads"], case["head_dim"]
        pages = sum(-(-c // PAGE) for c in ctx)
        moved = 4 * sum(ctx) * Hkv * D + 2 * 2 * len(ctx) * Hq * D + 4 * len(ctx) * (Hq + 1) + 4 * pages
        if case["append"]:
            moved += 2 * 4 * len(ctx) * Hkv * D
        return {"bytes": moved, "flops": 4 * sum(ctx) * Hq * D}
    if case["kind"] == "sdpa":
        B, Hq, Hkv, D = case["batch"], case["q_heads"], case["kv_heads"], case["head_dim"]
        Sq, Skv, kind = case["q_len"], case["kv_len"], case["mask"]
        keys = sum(_lengths(case)) if kind in ("pad", "pad_f16", "causal_f16") else B * Skv
        moved = 2 * 2 * B * Hq * Sq * D + 2 * 2 * keys * Hkv * D + (4 * B * Hq * Sq if case["lse"] else 0)
        moved += {"pad": B * Skv, "pad_f16": 2 * B * Skv, "causal_f16": 2 * B * Sq * Skv, "tail": Sq * Skv,
                  "bias_f32": 4 * Hq * Sq * Skv}.get(kind, 0)
        return {"bytes": moved, "flops": 4 * Hq * D * _pairs(case)}
    if case["kind"] == "relayout":
        n = math.prod(_host_size(case)) * (4 if case["dtype"] == "f32" else 2)
        return {"bytes": (6 if case["restick"] else 4) * n, "flops": 0}
    n = 2 * case["batch"] * case["kv_heads"] * case["length"] * case["head_dim"] * 2
    return {"bytes": 2 * n, "flops": 0}


def tolerance(case):
    if case["kind"] in ("relayout", "pages"):
        return "exact"
    # fp16 outputs of fp16 products with fp16 probabilities: about 4e-4 from the fp64 result.
    return {"rel": 2e-3, "max": 2e-2}


# ---------------------------------------------------------------- exact --

def _attend64(q, k, v, bias):
    """softmax(q k^T / sqrt(D) + bias) v of one KV head in fp64: q [R, D], k / v [S, D], bias
    broadcastable to [R, S] or None.  Returns (out, logsumexp)."""
    s = q.double() @ k.double().T / math.sqrt(q.shape[1])
    if bias is not None:
        s = s + bias
    lse = torch.logsumexp(s, dim=1)
    return torch.exp(s - lse[:, None]) @ v.double(), lse


def exact(case, seed):
    if case["kind"] == "paged":
        q, k, v, table, ctx, k_new, v_new = _paged_inputs(case, seed)
        Hq, Hkv, D = case["q_heads"], case["kv_heads"], case["head_dim"]
        g = Hq // Hkv
        if case["append"]:
            for b, n in enumerate(ctx):
                page, slot = int(table[b, (n - 1) // PAGE]), (n - 1) % PAGE
                k[page, :, :, slot, :] = k_new[b].view(Hkv, D // 64, 64)
                v[page, :, :, slot] = v_new[b]
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        lse = torch.empty(q.shape[:2], dtype=torch.float64, device="cuda")
        for b, n in enumerate(ctx):
            ids = table[b, :-(-n // PAGE)].long()
            kb = k[ids].permute(1, 0, 3, 2, 4).reshape(Hkv, -1, D)[:, :n]
            vb = v[ids].permute(1, 0, 3, 2).reshape(Hkv, -1, D)[:, :n]
            for h in range(Hkv):
                out[b, h * g:(h + 1) * g], lse[b, h * g:(h + 1) * g] = _attend64(q[b, h * g:(h + 1) * g], kb[h], vb[h], None)
        return (out, lse, k.double(), v.double()) if case["append"] else (out, lse)
    if case["kind"] != "sdpa":
        return None
    q, k, v, mask = _sdpa_inputs(case, seed)
    B, Hq, Sq, D = q.shape
    g = Hq // case["kv_heads"]
    if case["mask"] == "causal":
        mask = torch.ones((1, 1, Sq, k.shape[2]), dtype=torch.bool, device="cuda").tril()
    out = torch.empty((B, Sq, Hq, D), dtype=torch.float64, device="cuda").transpose(1, 2)
    lse = torch.empty((B, Hq, Sq), dtype=torch.float64, device="cuda")
    for b in range(B):
        for h in range(Hq):
            bias = None
            if mask is not None:
                m = mask[b % mask.shape[0], h % mask.shape[1]]
                bias = torch.zeros(m.shape, dtype=torch.float64, device="cuda").masked_fill_(~m, -math.inf) \
                    if m.dtype == torch.bool else m.double()
            out[b, h], lse[b, h] = _attend64(q[b, h], k[b, h // g], v[b, h // g], bias)
    return (out, lse) if case["lse"] else out
