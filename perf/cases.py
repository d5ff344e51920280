"""What a program that serves Qwen3-Next has this framework do, as cases to be timed.

A model has 48 layers, every fourth of them full attention: 16 query heads over 2 KV heads
of 256, a quantized KV cache (Q4K unless the user chooses Q8_0, F16 or BF16), and in between
Gated-DeltaNet layers whose state one token updates in place. One pass of a case is

- decode:  one token of a sequence: every full-attention layer appends the token's K and V
           and attends over all of its cache;
- chunk:   several tokens of one sequence: a prompt or a part of one (prefill), or a few
           drafted tokens that are verified at once (speculative decoding);
- token:   the whole of this framework's part of one token: the full-attention layers from
           their projections (norms, rope, append, attention, gated output projection) and
           the Gated-DeltaNet layers;
- serve:   one token of each of many sequences, every sequence with caches of its own;
- paged:   the same over sequences that share a pool of pages;
- restore: a saved prefix of a conversation is put back and its new suffix is appended.

`draw` takes more of each: caches from 32 to 131072 tokens, chunks from 2 to 4096, one to
32 sequences, all cache types.
"""
import math
import random

import torch

import paramecia_amd as pk
from paramecia_amd import workloads as W

H, KV, D = W.NUM_HEADS, W.NUM_KV_HEADS, W.HEAD_DIM
ROW_BYTES = {"q4k": 144, "q8_0": 272, "f16": 512, "bf16": 512}
W_TYPE = {"q4k": pk.WTYPE_Q4K, "q5k": pk.WTYPE_Q5K, "q6k": pk.WTYPE_Q6K}
W_BYTES = {"q4k": 144, "q5k": 176, "q6k": 210}
OUTLIERS = (11, 70, 101, 163, 240)  # channels of K and V that a trained model has far larger


def listed():
    return [
        # the first words of a conversation: one layer, a cache of a few dozen tokens
        dict(name="decode_start", kind="decode", quant="q4k", layers=1, batch=1, cached=97, graph=False),
        # a short chat in the finer format, its token captured once as a serving loop does
        dict(name="decode_q8_4k", kind="decode", quant="q8_0", layers=12, batch=1, cached=4096, graph=True),
        # an agent far into a repository: the longest context the framework is quoted on
        dict(name="decode_q4k_128k", kind="decode", quant="q4k", layers=12, batch=1, cached=131072, graph=False),
        # a user who wants an unquantized cache
        dict(name="decode_f16_12k", kind="decode", quant="f16", layers=12, batch=1, cached=12289, graph=False),
        # an ordinary chat's token through all 48 layers, captured once
        dict(name="token_q4k_6k", kind="token", quant="q4k", wo="q4k", layers=48, batch=1, cached=6001, graph=True),
        # four drafted tokens and the last accepted one, verified in one pass
        dict(name="verify_q4k_20k", kind="chunk", quant="q4k", layers=12, batch=1, cached=20011, length=5, prep=False),
        # a first prompt of ragged length, from the projections to the output projection
        dict(name="prompt_q4k_4k", kind="chunk", quant="q4k", layers=1, batch=1, cached=0, length=4001, prep=True),
        # the next 512 tokens of a long prompt
        dict(name="chunk_q4k_16k", kind="chunk", quant="q4k", layers=1, batch=1, cached=16384, length=512, prep=False),
        # the same in the finer format, ragged
        dict(name="chunk_q8_8k", kind="chunk", quant="q8_0", layers=1, batch=1, cached=8195, length=509, prep=False),
        # a serving batch of contexts between 1k and 64k tokens
        dict(name="serve_q4k_16", kind="serve", quant="q4k", layers=4, seqs=16, least=1024, most=65536, spread=1),
        # a busier server with shorter contexts in shared pages
        dict(name="paged_q4k_24", kind="paged", quant="q4k", layers=4, seqs=24, least=300, most=12000, spread=2, page=1024),
        # going back to a long conversation that was put aside
        dict(name="restore_q4k_64k", kind="restore", quant="q4k", layers=16, cached=65536, suffix=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = {c["name"]: _cost(c) for c in listed()}
    while True:
        kind = rng.choice(["decode", "decode", "chunk", "chunk", "chunk", "serve", "paged", "token", "restore"])
        quant = rng.choice(["q4k", "q4k", "q4k", "q8_0", "f16", "bf16"])
        if kind == "decode":
            c = dict(kind=kind, quant=quant, layers=rng.choice([1, 4, 12]), batch=rng.choice([1, 1, 1, 2, 4]),
                     cached=_log(rng, 32, 131072), graph=rng.random() < 0.4)
        elif kind == "chunk":
            c = dict(kind=kind, quant=quant, layers=1, batch=rng.choice([1, 1, 1, 2]), cached=_log(rng, 1, 65536) - 1,
                     length=rng.choice([_log(rng, 2, 16), _log(rng, 16, 4096)]), prep=rng.random() < 0.4)
        elif kind in ("serve", "paged"):
            least = _log(rng, 32, 8192)
            c = dict(kind=kind, quant=rng.choice(["q4k", "q4k", "q8_0"]), layers=rng.choice([1, 4]), seqs=_log(rng, 2, 32),
                     least=least, most=_log(rng, least, 65536), spread=rng.randrange(1000))
            if kind == "paged":
                c["page"] = 1 << rng.randrange(6, 13)
        elif kind == "token":
            c = dict(kind=kind, quant="q4k", wo=rng.choice(["q4k", "q5k", "q6k"]), layers=rng.choice([4, 48]),
                     batch=rng.choice([1, 1, 2]), cached=_log(rng, 32, 32768), graph=rng.random() < 0.5)
        else:
            c = dict(kind=kind, quant=rng.choice(["q4k", "q8_0"]), layers=rng.choice([4, 8, 16]), cached=_log(rng, 64, 65536),
                     suffix=_log(rng, 1, 1024))
        cost = _cost(c)
        limit = most["decode_f16_12k"] if c["quant"] in ("f16", "bf16") else most["decode_q4k_128k"]
        if cost["bytes"] <= limit["bytes"] and cost["flops"] <= most["chunk_q4k_16k"]["flops"]:
            if c["quant"] not in ("f16", "bf16") or kind == "decode" or cost["flops"] <= 3e9:
                return c


# ------------------------------------------------------------------ what a pass needs
def _lengths(c):
    r = random.Random(c["spread"])
    return [_log(r, c["least"], c["most"]) for _ in range(c["seqs"])]


def _cost(c):
    """Bytes (inputs and weights read once, results written once) and multiply-add operations."""
    rb, kind = 2 * KV * ROW_BYTES[c["quant"]], c["kind"]
    if kind == "restore":
        full = c["layers"] // 4
        state = 4 * (W.DN_HEADS * W.DN_DK * W.DN_DV + W.DN_CONV_DIM * (W.DN_CONV_K - 1) + W.DN_HEADS)
        back = full * c["cached"] * rb + (c["layers"] - full) * state
        return {"bytes": 2.0 * back + full * c["suffix"] * (rb + 2 * 4 * KV * D), "flops": 0.0}
    lens = _lengths(c) if kind in ("serve", "paged") else [c["cached"]] * c["batch"]
    l = c.get("length", 1)
    layers = c["layers"] // 4 if kind == "token" else c["layers"]
    new = l * len(lens)
    bytes_ = layers * (sum(lens) * rb + new * (rb + 2 * 4 * KV * D + 2 * 4 * H * D))
    flops = layers * 4.0 * H * D * sum(l * n + l * (l + 1) // 2 for n in lens)
    if kind == "token" or c.get("prep"):
        bytes_ += layers * (H * D // 256 * W.HIDDEN * W_BYTES[c.get("wo", "q4k")] + new * 4 * (H * D + W.HIDDEN))
        flops += layers * 2.0 * new * H * D * W.HIDDEN
    if kind == "token":
        dn = (c["layers"] - layers) * c["batch"] * W.DN_HEADS
        bytes_ += dn * 4.0 * (2 * W.DN_DK * W.DN_DV + 4 * W.DN_DV + 4)
        flops += dn * 8.0 * W.DN_DK * W.DN_DV
    return {"bytes": float(bytes_), "flops": flops}


def work(case):
    return _cost(case)


def tolerance(case):
    # Restored and appended bytes are whole numbers, and restored states are copies.
    if case["kind"] == "restore":
        return "exact"
    # Attention, projections and states in 32 bits (matrix operands as pairs of 16 bits); cache
    # bytes are exact. Against 64 bits the attention is off by up to 3.2e-6 here, and from the
    # projections by up to 1.6e-5: the norm leaves keys of a few large channels, whose scores
    # reach the tens, so that a rounding of the prepared q weighs as much more.
    return {"rel": 5e-5 if case["kind"] == "token" or case.get("prep") else 1e-5}


# ------------------------------------------------------------------ inputs
def _gen(seed, *at):
    g = torch.Generator(device="cuda")
    x = seed & 0x7FFFFFFF
    for a in at:
        x = (x * 1000003 + a + 1) & 0x7FFFFFFFFFFF
    g.manual_seed(x)
    return g


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _kv(seed, layer, seq, b, n, projected=False):
    """Keys and values as the projections and norms leave them: channels of unlike sizes, five
    of them far larger. [b, KV, n, D], or [b, n, KV, D] for projections still to be prepared."""
    g = _gen(seed, layer, seq, 1)
    size = torch.exp(0.4 * _normal(g, 2, D))
    size[:, list(OUTLIERS)] *= 6.0
    shape = (b, n, KV, D) if projected else (b, KV, n, D)
    return _normal(g, *shape).mul_(size[0]), _normal(g, *shape).mul_(size[1])


def _new(seed, layer, c, n, b):
    """A layer's new tokens: q, k, v, the output gate, and the norms' weights."""
    g = _gen(seed, layer, 0, 2)
    projected = c["kind"] == "token" or bool(c.get("prep"))
    k, v = _kv(seed, layer, 1 << 20, b, n, projected)
    d = {"q": _normal(g, b, n, H, D), "k": k, "v": v}
    if projected:
        d["gate"] = _normal(g, b, n, H * D)
        d["q_alpha"], d["k_alpha"] = 1.0 + 0.2 * _normal(g, D), 1.0 + 0.2 * _normal(g, D)
    return d


def _weights(seed, layer, wo):
    """The output projection of a GGUF file: random codes under plausible block scales."""
    g = _gen(seed, layer, 0, 3)
    nb = W.HIDDEN * H * D // 256
    w = torch.randint(0, 256, (nb, W_BYTES[wo]), generator=g, device="cuda", dtype=torch.uint8)
    d = (_normal(g, nb, 2).abs() + 0.125) * 1e-4
    d = d.half().view(torch.uint8).view(nb, 4)
    if wo == "q6k":
        w[:, 208:210] = d[:, :2]
    else:
        w[:, :4] = d
    return w.view(-1)


def _linear(seed, layer, b):
    """A Gated-DeltaNet layer's state and one token of it."""
    g, hd, d = _gen(seed, layer, 0, 4), W.DN_HEADS, W.DN_DV
    return {"ssm": _normal(g, b, hd, d, d) * 0.02, "conv": _normal(g, b, W.DN_CONV_DIM, W.DN_CONV_K - 1),
            "offset": _normal(g, b, hd), "q": _normal(g, b, 1, hd, d), "k": _normal(g, b, 1, hd, d), "v": _normal(g, b, 1, hd, d),
            "gate": -torch.nn.functional.softplus(_normal(g, b, 1, hd)), "beta": _normal(g, b, 1, hd)}


# ------------------------------------------------------------------ prepare
class _Bytes:
    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "|u1", "data": (ptr, False), "version": 3, "strides": None}


def _held(cache, n):
    """The cache's first n tokens as packed K and V bytes, eight to a value; each tensor keeps the
    cache that owns its memory alive."""
    old = cache.seq_len
    cache.set_len(n)
    kp, vp, size, _ = cache.get_kv_storage()
    cache.truncate(old)
    both = [torch.as_tensor(_Bytes(p, size), device="cuda").view(torch.int64) for p in (kp, vp)]
    for t in both:
        t.cache = cache
    return both


def _capture(s):
    """The pass as a HIP graph, as a serving loop keeps one per batch size."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _pass(s)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            s["outs"] = _pass(s)
    torch.cuda.current_stream().wait_stream(side)
    s["graph"] = g


def prepare(case, seed):
    c = dict(case)
    kind, quant = c["kind"], pk.KvCacheQuantization.from_str(c["quant"])
    s = {"case": c, "graph": None}
    if kind in ("decode", "chunk", "token"):
        b, cached, l = c["batch"], c["cached"], c.get("length", 1)
        full = range(c["layers"] // 4) if kind == "token" else range(c["layers"])
        s["full"], s["in"], s["kv"] = [], [], []
        rope = pk.RotaryEmbedding(W.N_ROT, cached + l, W.ROPE_THETA) if kind == "token" or c.get("prep") else None
        for i in full:
            at = pk.FullAttentionKv(H, KV, D, cached + l, quant)
            cache = at._ensure(b)
            if cached:
                k, v = _kv(seed, i, 0, b, cached)
                cache.append_quantized(k, v)
            n = _new(seed, i, c, l, b)
            if rope is not None:
                n["prep"] = pk.QkPrep(n["q_alpha"], n["k_alpha"], W.RMS_EPS, rope)
                n["wo"] = _weights(seed, i, c.get("wo", "q4k"))
            s["kv"] += _held(cache, cached + l)
            s["full"].append(at)
            s["in"].append(n)
        if kind == "token":
            lin = [_linear(seed, i, b) for i in range(c["layers"] - len(full))]
            s["ssm"] = torch.stack([x.pop("ssm") for x in lin])
            s["offset"] = torch.stack([x.pop("offset") for x in lin])
            s["lin"], s["lin_in"] = [], lin
            for i, x in enumerate(lin):
                la = pk.LinearAttentionState(W.DN_DV ** -0.5, W.RMS_EPS, W.DN_CONV_DIM, W.DN_CONV_K)
                la.recurrent_state = pk.RecurrentState(s["ssm"][i], x.pop("conv"), s["offset"][i])
                s["lin"].append(la)
    elif kind == "serve":
        s["lens"] = _lengths(c)
        s["caches"], s["in"] = [], []
        for i in range(c["layers"]):
            row = []
            for j, n in enumerate(s["lens"]):
                cache = pk.PreallocatedQuantizedKvCache(1, KV, n + 1, D, quant)
                cache.append_quantized(*_kv(seed, i, j, 1, n))
                row.append(cache)
            x = _new(seed, i, c, 1, c["seqs"])
            s["caches"].append(row)
            s["in"].append((x["k"].view(-1, KV, D), x["v"].view(-1, KV, D), x["q"].view(-1, H, D)))
    elif kind == "paged":
        s["lens"] = _lengths(c)
        pages = sum(n // c["page"] + 1 for n in s["lens"])
        s["pools"], s["seqs"], s["in"] = [], [], []
        for i in range(c["layers"]):
            pool = pk.PagedKvPool(KV, D, c["page"], pages, quant)
            row = []
            for j, n in enumerate(s["lens"]):
                sq = pool.sequence()
                sq.append_quantized(*_kv(seed, i, j, 1, n))
                row.append(sq)
            x = _new(seed, i, c, 1, c["seqs"])
            s["pools"].append(pool)
            s["seqs"].append(row)
            s["in"].append((x["k"], x["v"], x["q"].view(-1, H, D)))
    else:
        model = pk.ModelKvState(c["layers"], W.FULL_INTERVAL, H, KV, D, c["cached"] + c["suffix"], quant)
        s["suffix"] = []
        for i, layer in enumerate(model.layers):
            if isinstance(layer, pk.FullAttentionKv):
                layer._ensure(1).append_quantized(*_kv(seed, i, 0, 1, c["cached"]))
                s["suffix"].append(_kv(seed, i, 1, 1, c["suffix"]))
            else:
                x = _linear(seed, i, 1)
                layer.recurrent_state = pk.RecurrentState(x["ssm"], x["conv"], x["offset"])
        s["model"], s["prefix"] = model, model.save_prefix_cache(list(range(c["cached"])))
        s["kv"] = []
        for layer in model.full_layers():
            s["kv"] += _held(layer.quantized_cache, c["cached"] + c["suffix"])
    if c.get("graph"):
        keep = (s["ssm"].clone(), s["offset"].clone()) if kind == "token" else None
        _capture(s)
        if keep is not None:  # the warm-up has moved the states
            s["ssm"].copy_(keep[0])
            s["offset"].copy_(keep[1])
    return s


# ------------------------------------------------------------------ run
def _pass(s):
    c = s["case"]
    kind = c["kind"]
    if kind in ("decode", "chunk", "token"):
        at = c["cached"]  # the sequence goes on from here: a repeated pass rewinds its tokens
        outs = []
        for layer, n in zip(s["full"], s["in"]):
            if "prep" in n:
                o = layer.forward_projected(n["q"], n["k"], n["v"], at, n["prep"])
                o = pk.gated_o_proj(o, n["gate"], n["wo"], W.HIDDEN, W_TYPE[c.get("wo", "q4k")])
            else:
                o = layer.forward(n["q"], n["k"], n["v"], at)
            outs.append(o)
        if kind == "token":
            for layer, x in zip(s["lin"], s["lin_in"]):
                outs.append(layer.delta_net_autoregressive(x["q"], x["k"], x["v"], x["gate"], x["beta"]))
            return outs + [s["ssm"], s["offset"]]
        return outs + s["kv"]
    if kind == "serve":
        outs = []
        for row, (k, v, q) in zip(s["caches"], s["in"]):
            for cache, n in zip(row, s["lens"]):
                cache.truncate(n)
            outs.append(pk.append_attend_batched(row, k, v, q, W.SCALE))
        return outs
    if kind == "paged":
        outs = []
        for pool, row, (k, v, q) in zip(s["pools"], s["seqs"], s["in"]):
            for sq, n in zip(row, s["lens"]):
                sq.truncate(n)
            outs.append(pool.append_decode_batched(row, k, v, q, W.SCALE))
        return outs
    model = s["model"]
    model.restore_prefix_cache(s["prefix"])
    for layer, (k, v) in zip(model.full_layers(), s["suffix"]):
        layer.quantized_cache.append_quantized(k, v, c["cached"])
    outs = list(s["kv"])
    for layer in model.layers:
        if isinstance(layer, pk.LinearAttentionState):
            r = layer.recurrent_state
            outs += [r.ssm_state, r.conv_state, r.gate_cumsum_offset]
    return outs


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        return state["outs"]
    return _pass(state)


# ------------------------------------------------------------------ the same in 64 bits
def _over(a, b):
    """a / b rounded once: torch multiplies by a reciprocal where one side is a plain number."""
    full = b if torch.is_tensor(b) else a
    return torch.div(*(x if torch.is_tensor(x) else torch.full_like(full, x) for x in (a, b)))


def _round_away(v):
    r = torch.trunc(v)
    return r + torch.sign(v) * ((v - r).abs() >= 0.5)


def _scale_min(sc):
    """The eight 6-bit scales and mins of a k-quant header [N, 12]."""
    sc = sc.int()
    lo, hi = sc[:, :4], sc[:, 4:8]
    s = torch.cat([lo & 63, (sc[:, 8:] & 15) | ((lo >> 6) << 4)], 1)
    m = torch.cat([hi & 63, (sc[:, 8:] >> 4) | ((hi >> 6) << 4)], 1)
    return s, m


def _q4k(x):
    """What a Q4K cache holds of the rows x [N, 256]: GGML's fit (five passes, sums in order)."""
    t = x.view(-1, 32).t().contiguous()  # an element a row, so that sums go element by element
    low, high = t.amin(0).clamp(max=0), t.amax(0)
    iscale = _over(15.0, high - low)
    scale, old, live = _over(1.0, iscale), torch.zeros_like(t), torch.ones_like(low, dtype=torch.bool)
    for _ in range(5):
        lev = _round_away(iscale * (t - low)).clamp_(0, 15)
        terms, total = (t - low) * lev, torch.zeros_like(low)
        for i in range(32):
            total = total + terms[i]
        s = total / (lev * lev).sum(0)
        terms, total = t - s * lev, torch.zeros_like(low)
        for i in range(32):
            total = total + terms[i]
        m = (total / 32.0).clamp(max=0)
        scale, low, iscale = torch.where(live, s, scale), torch.where(live, m, low), torch.where(live, _over(1.0, s), iscale)
        live &= (lev != old).any(0)
        old = lev
    scale, least = scale.view(-1, 8), -low.view(-1, 8)
    top, top_m = scale.amax(1, keepdim=True).clamp(min=0), least.amax(1, keepdim=True).clamp(min=0)
    inv = torch.where(top > 0, _over(63.0, top), 0.0)
    inv_m = torch.where(top_m > 0, _over(63.0, top_m), 0.0)
    ls, lm = _round_away(inv * scale).clamp(max=63), _round_away(inv_m * least).clamp(max=63)
    d, dm = _over(top, 63.0).half().float() * ls, _over(top_m, 63.0).half().float() * lm
    x = x.view(-1, 8, 32)
    lev = _round_away((x + dm[:, :, None]) / d[:, :, None]).clamp(0, 15)
    lev = torch.where(d[:, :, None] != 0, lev, torch.zeros_like(lev))
    return (d.double()[:, :, None] * lev.double() - dm.double()[:, :, None]).view(-1, 256)


def _stored(x, quant):
    """The cache's values of x [..., 256] f32, in 64 bits."""
    flat, out = x.reshape(-1, D), torch.empty(x.shape, dtype=torch.float64, device=x.device)
    for i in range(0, flat.shape[0], 1 << 16):
        r = flat[i:i + (1 << 16)]
        if quant == "q4k":
            y = _q4k(r)
        elif quant == "q8_0":
            b = r.reshape(-1, 32)
            d = _over(b.abs().amax(1, keepdim=True), 127.0)
            y = (_round_away(b * torch.where(d > 0, _over(1.0, d), 0.0)).double() * d.half().double()).view(-1, D)
        else:
            y = (r.half() if quant == "f16" else r.bfloat16()).double()
        out.view(-1, D)[i:i + (1 << 16)] = y
    return out


def _attention(q, k, v, cached):
    """q [b, l, H, D], k, v [b, KV, S, D] in 64 bits; query i sees the keys up to cached + i."""
    b, l = q.shape[:2]
    out = torch.empty_like(q)
    seen = torch.arange(k.shape[2], device="cuda")
    for n in range(b):
        for h in range(H):
            kh, vh = k[n, h // (H // KV)], v[n, h // (H // KV)]
            for i in range(0, l, 512):
                at = torch.arange(i, min(l, i + 512), device="cuda")
                z = (q[n, at, h] @ kh.t() * W.SCALE).clamp_(-100, 100)
                z.masked_fill_(seen[None, :] > cached + at[:, None], -math.inf)
                out[n, at, h] = torch.softmax(z, 1) @ vh
    return out


def _prepared(x, alpha, cached, dtype=torch.float64):
    """RMS norm and rotary embedding of x [b, l, heads, D]. Keys take 32-bit steps, with the norm's
    sum in order: the cache's codes follow from that rounding."""
    x, alpha = x.to(dtype), alpha.to(dtype)
    sq, total = x.square(), torch.zeros_like(x[..., 0])
    for i in range(D):
        total = total + sq[..., i]
    x = _over(x, torch.sqrt(total / D + W.RMS_EPS)[..., None]) * alpha
    half = W.N_ROT // 2
    # the model defines its angles as 32-bit products of position and frequency
    power = torch.pow(torch.tensor(W.ROPE_THETA, dtype=torch.float64), torch.arange(half, dtype=torch.float64) * 2 / W.N_ROT)
    pos = torch.arange(cached, cached + x.shape[1], dtype=torch.float32)
    ang = (pos[:, None] * _over(1.0, power.float())[None, :]).double().to(x.device)[None, :, None, :]
    cos, sin = (t.float().to(dtype) for t in (ang.cos(), ang.sin()))
    a, b = x[..., :half], x[..., half:2 * half]
    return torch.cat([a * cos - b * sin, a * sin + b * cos, x[..., 2 * half:]], -1)


def _weight_values(w, wo):
    w = w.view(-1, W_BYTES[wo])
    f16 = lambda x: x.contiguous().view(torch.float16).double()  # noqa: E731
    if wo == "q6k":
        lo, hi = w[:, :128].int(), w[:, 128:192].int()
        sc = w[:, 192:208].contiguous().view(torch.int8).double()
        parts = []
        for n in range(2):
            a, h = lo[:, 64 * n:64 * n + 64], hi[:, 32 * n:32 * n + 32]
            parts += [(a[:, :32] & 15) | ((h & 3) << 4), (a[:, 32:] & 15) | (((h >> 2) & 3) << 4),
                      (a[:, :32] >> 4) | (((h >> 4) & 3) << 4), (a[:, 32:] >> 4) | (((h >> 6) & 3) << 4)]
        q = torch.cat(parts, 1).double() - 32
        y = f16(w[:, 208:210]) * (q.view(-1, 16, 16) * sc[:, :, None]).view(-1, 256)
    else:
        s, m = _scale_min(w[:, 4:16])
        qs = w[:, -128:].int().view(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).view(-1, 8, 32)
        if wo == "q5k":
            fifth = (w[:, 16:48].int()[:, None, :] >> torch.arange(8, device=w.device, dtype=torch.int32)[None, :, None]) & 1
            q = q + 16 * fifth
        y = f16(w[:, :2])[:, :, None] * (s[:, :, None] * q).double() - f16(w[:, 2:4])[:, :, None] * m.double()[:, :, None]
    return y.reshape(W.HIDDEN, H * D)


def _delta(x):
    """One Gated-DeltaNet token: its output, the new state and gate offset."""
    x = {k: v.double() for k, v in x.items()}
    unit = lambda t: t / torch.sqrt(t.square().sum(-1, keepdim=True) + W.RMS_EPS)  # noqa: E731
    q, k, v = unit(x["q"][:, 0]) * W.DN_DV ** -0.5, unit(x["k"][:, 0]), x["v"][:, 0]
    st = x["ssm"] * torch.exp(x["gate"][:, 0])[..., None, None]
    err = (v - (st * k[:, :, None, :]).sum(-1)) * torch.sigmoid(x["beta"][:, 0])[..., None]
    st = st + err[..., None] * k[:, :, None, :]
    return (st * q[:, :, None, :]).sum(-1)[:, None], st, x["offset"] + x["gate"][:, 0]


def exact(case, seed):
    c, outs = dict(case), []
    kind, quant = c["kind"], c["quant"]
    if kind == "restore":
        return None
    if kind in ("serve", "paged"):
        for i in range(c["layers"]):
            x = _new(seed, i, c, 1, c["seqs"])
            rows = []
            for j, n in enumerate(_lengths(c)):
                k, v = _kv(seed, i, j, 1, n)
                k, v = torch.cat([k, x["k"][j:j + 1]], 2), torch.cat([v, x["v"][j:j + 1]], 2)
                rows.append(_attention(x["q"][j:j + 1].double(), _stored(k, quant), _stored(v, quant), n)[0, 0])
            outs.append(torch.stack(rows))
        return outs
    b, l, cached = c["batch"], c.get("length", 1), c["cached"]
    for i in range(c["layers"] // 4 if kind == "token" else c["layers"]):
        x = _new(seed, i, c, l, b)
        q, kn, vn = x["q"].double(), x["k"], x["v"]
        if "gate" in x:
            q = _prepared(x["q"], x["q_alpha"], cached)
            kn = _prepared(kn, x["k_alpha"], cached, torch.float32).transpose(1, 2)
            vn = vn.transpose(1, 2)
        if cached:
            k, v = _kv(seed, i, 0, b, cached)
            kn, vn = torch.cat([k, kn], 2), torch.cat([v, vn], 2)
            del k, v
        o = _attention(q, _stored(kn, quant), _stored(vn, quant), cached).reshape(b, l, H * D)
        if "gate" in x:
            w = _weight_values(_weights(seed, i, c.get("wo", "q4k")), c.get("wo", "q4k"))
            o = (o * torch.sigmoid(x["gate"].double())) @ w.t()
        outs.append(o)
        del kn, vn
    if kind != "token":
        outs += [None] * (2 * c["layers"])
    else:
        lin = [_delta(_linear(seed, i, b)) for i in range(c["layers"] - c["layers"] // 4)]
        outs += [o for o, _, _ in lin]
        outs += [torch.stack([st for _, st, _ in lin]), torch.stack([g for _, _, g in lin])]
    return outs
