"""Workloads of the attention path, through the public entry points, for timing and comparison.

A case is one call (or one layer's step) as a serving loop makes it:

* ``decode``  -- ``paged_attention`` with one query token per sequence;
* ``mixed``   -- ``paged_attention`` over a ragged batch: prompt chunks of several query tokens
  (causal, over an already cached prefix) beside single-token rows;
* ``step``    -- one decode step of one layer: ``concatenate_to_cache`` with RoPE (one new token per
  sequence appended to its page) and the registered attention operation over the result;
* ``write``   -- a prompt's keys and values (and the rotation of its queries) into the cache pages.

Caches: unquantized fp16 / bf16 in the ``[num_blocks, page, Hkv, D]`` layout (the default cache type),
affine 4-bit and 8-bit pages (group 64), FP8 (E4M3) pages.  Sizes come from the benchmark
configurations (batch 32 with contexts of 512 to 4096, 8 contexts of 32768, four 512-token chunks
beside 28 decode rows), the default page of 16 tokens and the 128-token page of the benchmarks,
and head sizes 64, 128 and 256.
"""

from __future__ import annotations

import math
import zlib

import numpy as np
import torch

from easymlx_amd import (
    AffinePageCacheView,
    Fp8PageCacheView,
    OperationRegistry,
    PageCacheView,
    PageMetadata,
    RotaryEmbedding,
    paged_attention,
)

DEV = "cuda"
GROUP = 64


# ---------------------------------------------------------------- cases


def _decode(name, cache, seqs, lo, hi, hq, hkv, d, page, window=0):
    return dict(name=name, kind="decode", cache=cache, seqs=seqs, ctx_lo=lo, ctx_hi=hi, hq=hq, hkv=hkv, d=d, page=page,
                window=window)


def _mixed(name, cache, chunks, chunk, prior, rows, lo, hi, hq, hkv, d, page, window=0):
    return dict(name=name, kind="mixed", cache=cache, chunks=chunks, chunk=chunk, prior=prior, seqs=rows, ctx_lo=lo,
                ctx_hi=hi, hq=hq, hkv=hkv, d=d, page=page, window=window)


def listed():
    return [
        # one user, one token: the latency of a single request over the unquantized default cache
        _decode("decode_one_f16", "f16", 1, 1024, 1024, 32, 8, 64, 128),
        # a serving batch over the default cache: bf16, the default page of 16 tokens
        _decode("decode_bf16_p16", "bf16", 32, 512, 4096, 32, 8, 128, 16),
        # the benchmark's headline call: a serving batch over 4-bit pages
        _decode("decode_q4", "q4", 32, 512, 4096, 32, 8, 128, 128),
        # eight long documents over 4-bit pages, a large model's 64 query heads
        _decode("decode_q4_long", "q4", 8, 32768, 32768, 64, 8, 128, 128),
        # FP8 cache as PageCacheConfig allocates it by default (pages of 16 tokens), ragged contexts
        _decode("decode_fp8_p16", "fp8", 32, 300, 3500, 32, 8, 128, 16),
        # head size 256 over 8-bit pages: few kv heads, a small batch
        _decode("decode_q8_d256", "q8", 13, 200, 5000, 16, 4, 256, 64),
        # continuous batching over 4-bit pages: four prompt chunks beside 28 decoding sequences
        _mixed("mixed_q4", "q4", 4, 512, 2048, 28, 256, 4096, 32, 8, 128, 128),
        # the same step over the default cache
        _mixed("mixed_bf16_p16", "bf16", 4, 512, 2048, 28, 256, 4096, 32, 8, 128, 16),
        # 4-bit pages of the default size, odd chunks, a smaller batch
        _mixed("mixed_q4_p16", "q4", 3, 203, 700, 9, 50, 1500, 32, 8, 128, 16),
        # one prompt at head size 256 with a sliding window, nothing cached before it, no decode rows
        _mixed("prompt_f16_d256", "f16", 1, 1531, 0, 0, 1, 1, 16, 8, 256, 32, window=700),
        # one layer of a small batch's decode step: append with RoPE, then the registered operation
        dict(name="step_q4", kind="step", cache="q4", seqs=16, ctx_lo=100, ctx_hi=1000, hq=32, hkv=8, d=128, page=128,
             window=0),
        # four prompt chunks written to 4-bit pages, keys and queries rotated
        dict(name="write_q4", kind="write", cache="q4", seqs=4, tokens=512, hq=32, hkv=8, d=128, page=128, window=0),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["decode", "mixed", "step", "write"], [9, 8, 2, 2])[0]
    cache = rng.choices(["f16", "bf16", "q4", "q8", "fp8"], [3, 4, 5, 3, 3])[0]
    d = rng.choices([64, 128, 256], [2, 5, 1])[0]
    page = rng.choices([16, 32, 64, 128], [3, 1, 1, 3])[0]
    # query heads per kv head 1, 2, 3, 4, 7 and 8, over the kv heads a layer (or its share) has
    hq, hkv = rng.choice([(32, 8), (32, 8), (64, 8), (16, 8), (16, 16), (24, 8), (28, 4), (8, 2), (8, 1)])
    window = rng.choice([0, 0, 0, 0, rng.randint(100, 2000)])
    if kind == "write":
        seqs = rng.randint(1, 4)
        return dict(kind=kind, cache=cache, seqs=seqs, tokens=_logu(rng, 2, 1024), hq=hq, hkv=hkv, d=d, page=page,
                    window=0)
    # at most the keys and values of the largest listed decode (as unquantized values)
    budget = 72_000 * 8 * 128
    if kind in ("decode", "step"):
        seqs = _logu(rng, 1, 96)
        top = max(16, min(32768, budget // (seqs * hkv * d)))
        hi = _logu(rng, 16, top)
        lo = max(1, int(hi * rng.uniform(0.1, 1.0)))
        return dict(kind=kind, cache=cache, seqs=seqs, ctx_lo=lo, ctx_hi=hi, hq=hq, hkv=hkv, d=d, page=page,
                    window=window if kind == "decode" else 0)
    chunks, chunk, prior = rng.randint(1, 4), _logu(rng, 2, 700), rng.choice([0, _logu(rng, 16, 1500)])
    # the matrix work of a chunk stays below a third of the largest listed mixed step
    while chunks * chunk * (prior + chunk) * hq * d > 4 * 512 * 1500 * 32 * 128 // 3:
        chunk = max(2, chunk // 2)
        prior //= 2
    rows = rng.choice([0, rng.randint(1, 28)])
    hi = _logu(rng, 16, 2500)
    return dict(kind=kind, cache=cache, chunks=chunks, chunk=chunk, prior=prior, seqs=rows,
                ctx_lo=max(1, int(hi * rng.uniform(0.1, 1.0))), ctx_hi=hi, hq=hq, hkv=hkv, d=d, page=page,
                window=window)


# ---------------------------------------------------------------- inputs


def _lengths(case):
    """``(query lengths, key lengths)`` of every sequence, from the case alone."""
    rng = np.random.default_rng(zlib.crc32(repr(sorted((k, v) for k, v in case.items() if k != "name")).encode()))
    if case["kind"] == "write":
        return [case["tokens"]] * case["seqs"], [case["tokens"]] * case["seqs"]
    rows = [int(x) for x in rng.integers(case["ctx_lo"], case["ctx_hi"] + 1, size=case["seqs"])]
    if case["kind"] != "mixed":
        return [1] * len(rows), rows
    prior = [int(x) for x in rng.integers(0, case["prior"] + 1, size=case["chunks"])]
    return [case["chunk"]] * case["chunks"] + [1] * len(rows), [p + case["chunk"] for p in prior] + rows


def _dtype(case):
    return torch.bfloat16 if case["cache"] == "bf16" else torch.float16


def _inputs(case, seed):
    """Queries, keys and values (logical order), the block table of a shuffled pool, slots and lengths."""
    qlens, kvl = _lengths(case)
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    hq, hkv, d, page = case["hq"], case["hkv"], case["d"], case["page"]
    n = sum(kvl)
    dt = _dtype(case)
    # keys and values with per-channel gains of 0.5 to 4, as trained projections have
    gains = torch.rand((2, 1, hkv, d), generator=g, device=DEV) * 3.5 + 0.5
    q = torch.randn((sum(qlens), hq, d), generator=g, device=DEV).to(dt)
    k = (torch.randn((n, hkv, d), generator=g, device=DEV) * gains[0]).to(dt)
    v = (torch.randn((n, hkv, d), generator=g, device=DEV) * gains[1]).to(dt)
    pages = [-(-(x + (case["kind"] == "step")) // page) for x in kvl]  # a step appends one token
    pool = sum(pages)
    perm = np.random.default_rng(seed).permutation(pool).astype(np.int32)
    tables = np.full((len(kvl), max(pages)), -1, np.int32)
    at = 0
    for i, p in enumerate(pages):
        tables[i, :p] = perm[at:at + p]
        at += p
    slot = np.concatenate([tables[i, np.arange(x) // page].astype(np.int64) * page + np.arange(x) % page
                           for i, x in enumerate(kvl)])
    return dict(q=q, k=k, v=v, pool=pool, tables=tables, slot=torch.from_numpy(slot).to(DEV), qlens=qlens, kvl=kvl)


def _affine(x, bits):
    """Affine codes and fp16 scale / bias per 64-value group of ``x [..., D]``."""
    xf = x.float().unflatten(-1, (-1, GROUP))
    lo, hi = xf.amin(-1, keepdim=True), xf.amax(-1, keepdim=True)
    neg = lo.abs() > hi.abs()
    step = ((hi - lo) / (2 ** bits - 1)).clamp_min(1e-7)
    scale = torch.where(neg, step, -step).to(torch.float16)
    bias = torch.where(neg, lo, hi).to(torch.float16)
    code = ((xf - bias.float()) / scale.float()).round().clamp(0, 2 ** bits - 1).to(torch.uint8)
    return code.flatten(-2), scale.squeeze(-1), bias.squeeze(-1)


def _fp8(x):
    """E4M3 codes of ``x / scale`` with one scale, ``max|x| / 240``."""
    scale = float(x.abs().max()) / 240.0
    return (x.float() / scale).to(torch.float8_e4m3fn).view(torch.uint8), scale


def _scatter(x, slot, pool, page):
    out = torch.zeros((pool * page,) + tuple(x.shape[1:]), dtype=x.dtype, device=DEV)
    out[slot] = x
    return out.unflatten(0, (pool, page))


def _words(nib, bits):
    """Bytes (8-bit) or nibbles (4-bit, low first) of the last axis as int32 words."""
    if bits == 4:
        nib = nib[..., 0::2] | (nib[..., 1::2] << 4)
    return nib.contiguous().view(torch.int32)


def _view(case, inp):
    """The cache view holding the inputs' keys and values, as an engine's earlier writes left it."""
    hkv, d, page, pool = case["hkv"], case["d"], case["page"], inp["pool"]
    tables = torch.from_numpy(inp["tables"]).to(DEV)
    lens = torch.tensor(inp["kvl"], dtype=torch.int32, device=DEV)
    common = dict(block_tables=tables, kv_lens=lens, block_size=page, num_kv_heads=hkv, head_dim=d)
    slot, cache = inp["slot"], case["cache"]
    empty = case["kind"] == "write"
    k, v = (inp["k"][:0], inp["v"][:0]) if empty else (inp["k"], inp["v"])
    slot = slot[:0] if empty else slot
    if cache in ("f16", "bf16"):
        return PageCacheView(key_cache=_scatter(k, slot, pool, page), value_cache=_scatter(v, slot, pool, page),
                             **common)
    if cache == "fp8":
        arrays, scales = [], []
        for x in (k, v):
            c, s = _fp8(x) if x.numel() else (x.to(torch.uint8), 0.0)
            arrays.append(_scatter(c, slot, pool, page))
            scales.append(torch.full((pool,), s, dtype=torch.float32, device=DEV))
        return Fp8PageCacheView(key_cache=arrays[0], value_cache=arrays[1], k_scales=scales[0], v_scales=scales[1],
                                **common)
    bits = 4 if cache == "q4" else 8
    out = {}
    for name, x in (("k", k), ("v", v)):
        if x.numel():
            code, sc, bi = _affine(x, bits)
        else:
            code, sc = x.to(torch.uint8), x[..., :: GROUP]
            bi = sc
        code = _scatter(code, slot, pool, page).permute(0, 2, 1, 3)  # [pool, Hkv, page, D]
        if name == "k":
            out["k_codes"] = _words(code, bits)
        else:  # tiles of T tokens, dim-major inside; 4-bit words hold token 2j, 2j + 1 at nibbles j, j + 4
            t = min(page, 256 // bits)
            code = code.unflatten(2, (page // t, t)).transpose(3, 4)  # [pool, Hkv, page/T, D, T]
            if bits == 4:
                code = code.unflatten(-1, (t // 8, 8))[..., [0, 2, 4, 6, 1, 3, 5, 7]].flatten(-2)
            out["v_codes"] = _words(code, bits)
        out[name + "_scales"] = _scatter(sc, slot, pool, page).permute(0, 2, 3, 1).contiguous()
        out[name + "_biases"] = _scatter(bi, slot, pool, page).permute(0, 2, 3, 1).contiguous()
    return AffinePageCacheView(**out, bits=bits, group_size=GROUP, **common)


def _stored(case, k, v):
    """The values the pages hold for tokens ``k``, ``v``, in 64 bits."""
    if case["cache"] in ("f16", "bf16"):
        return k.double(), v.double()
    out = []
    for x in (k, v):
        if case["cache"] == "fp8":
            c, s = _fp8(x)
            out.append(c.view(torch.float8_e4m3fn).double() * float(np.float32(s)))
        else:
            c, s, b = _affine(x, 4 if case["cache"] == "q4" else 8)
            out.append((c.double().unflatten(-1, (-1, GROUP)) * s.double()[..., None]
                        + b.double()[..., None]).flatten(-2))
    return out


# ---------------------------------------------------------------- the calls


def _rope(case):
    return RotaryEmbedding.llama3(case["d"], base=500000.0)


def _new_tokens(case, inp, seed):
    """A step's new token of every sequence (pre-rotation keys), drawn after the cached ones."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed + 1)
    shape = (case["seqs"], case["hkv"], case["d"])
    return [torch.randn(shape, generator=g, device=DEV).to(_dtype(case)) for _ in range(2)]


def prepare(case, seed):
    inp = _inputs(case, seed)
    view = _view(case, inp)
    state = dict(case=case, view=view, q=inp["q"],
                 qsl=torch.tensor(np.concatenate([[0], np.cumsum(inp["qlens"])]), dtype=torch.int32, device=DEV))
    if case["kind"] in ("step", "write"):
        if case["kind"] == "step":
            state["k"], state["v"] = _new_tokens(case, inp, seed)
        else:
            view.kv_lens.zero_()
            state["k"], state["v"] = inp["k"], inp["v"]
        state["lens"] = view.kv_lens.clone()  # the scheduler's lengths before the step
        state["ids"] = tuple(range(len(inp["kvl"])))
        state["qlens"] = tuple(inp["qlens"])
        state["md"] = PageMetadata(query_start_loc=state["qsl"], is_single_token_decode=case["kind"] == "step",
                                   slot_ids=state["ids"])
        state["rope"] = _rope(case)
        state["op"] = OperationRegistry.create("unified_attention")
    return state


def run(state):
    case, view = state["case"], state["view"]
    if case["kind"] in ("decode", "mixed"):
        kw = {}
        if view.is_affine:
            kw = dict(k_scales=view.k_scales, k_biases=view.k_biases, v_scales=view.v_scales, v_biases=view.v_biases,
                      bits=view.bits, group_size=view.group_size)
        elif case["cache"] == "fp8":
            kw = dict(k_scale=view.k_scales, v_scale=view.v_scales)
        return paged_attention(state["q"], view.key_cache, view.value_cache, view.block_tables, view.kv_lens,
                               state["qsl"], sliding_window=case["window"] or None,
                               single_token_decode=case["kind"] == "decode", **kw)
    view.kv_lens.copy_(state["lens"])  # the scheduler hands over every sequence's length
    q, k, v, md = view.concatenate_to_cache(state["q"], state["k"], state["v"], cache_metadata=state["md"],
                                            rope=state["rope"], slot_ids=state["ids"], query_lens=state["qlens"])
    out = [q]
    if case["kind"] == "step":
        out.append(state["op"](query=q, key=k, value=v, cache_metadata=md, cache_view=view).attention_outputs)
    return out + view.page_arrays()


# ---------------------------------------------------------------- what a pass cannot do without


def _kv_bytes(case):
    """Bytes of one token's key and value in one kv head."""
    d = case["d"]
    return {"f16": 4 * d, "bf16": 4 * d, "fp8": 2 * d, "q4": d + 8 * (d // GROUP),
            "q8": 2 * d + 8 * (d // GROUP)}[case["cache"]]


def _visible(case, ql, kl):
    """``(keys any row reads, (row, key) pairs)`` of a sequence with ``ql`` query rows over ``kl`` keys."""
    w = case["window"] or kl
    first = max(0, kl - ql + 1 - w)
    return kl - first, sum(min(w, kl - ql + i + 1) for i in range(ql))


def work(case):
    qlens, kvl = _lengths(case)
    row = 2 * case["hq"] * case["d"]
    per = _kv_bytes(case) * case["hkv"]
    if case["kind"] == "write":  # k, v and q read, pages and turned q written
        n = sum(qlens)
        return {"bytes": n * (2 * row + 4 * case["hkv"] * case["d"] + per), "flops": 0}
    keys = pairs = 0
    for ql, kl in zip(qlens, kvl):
        kl += case["kind"] == "step"
        a, b = _visible(case, ql, kl)
        keys += a
        pairs += b
    return {"bytes": 2 * sum(qlens) * row + keys * per, "flops": 4 * pairs * case["hq"] * case["d"]}


def tolerance(case):
    # attention: rounding of the 16-bit result (2^-12 / 2^-9 of a value) and of the operands a matrix
    # unit takes in 16 bits; the quantized pages themselves are the same on both sides
    if case["kind"] == "write" and case["cache"] not in ("f16", "bf16"):
        return "exact"  # codes, scales and rotated rows are defined bit for bit
    # (measured against 64 bits: fp16 2.0e-4 to 4.1e-4 with a largest difference of 3.8e-3, bf16 1.7e-3 and
    # 3.9e-3; four times that)
    return {"rel": 7e-3, "max": 1.6e-2} if case["cache"] == "bf16" else {"rel": 1.6e-3, "max": 1.5e-2}


# ---------------------------------------------------------------- 64 bits


def _attend(case, q, k, v, qlens, kvl):
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    hg = hq // hkv
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    qa = ka = 0
    for ql, kl in zip(qlens, kvl):
        kt = k[ka:ka + kl].permute(1, 2, 0).contiguous()  # [Hkv, D, kl]
        vs = v[ka:ka + kl].permute(1, 0, 2).contiguous()
        past = kl - ql
        for r0 in range(0, ql, 256):
            n = min(256, ql - r0)
            qs = q[qa + r0:qa + r0 + n].double().reshape(n, hkv, hg, d).permute(1, 2, 0, 3).reshape(hkv, hg * n, d)
            s = torch.bmm(qs, kt) / math.sqrt(d)
            pos = past + r0 + torch.arange(n, device=DEV)
            t = torch.arange(kl, device=DEV)
            seen = t[None] <= pos[:, None]
            if case["window"]:
                seen &= t[None] > pos[:, None] - case["window"]
            s.masked_fill_(~seen.repeat(hg, 1)[None], -math.inf)
            o = torch.bmm(torch.softmax(s, -1), vs)
            out[qa + r0:qa + r0 + n] = o.reshape(hkv, hg, n, d).permute(2, 0, 1, 3).reshape(n, hq, d)
        qa += ql
        ka += kl
    return out


def _llama3_inv(d):
    """Inverse frequencies of the piecewise scaled rotation (factor 8, 1 / 4, 8192 positions), fp32."""
    i = torch.arange(0, d, 2, dtype=torch.float32)
    f = torch.pow(torch.tensor(500000.0), i / d)
    wl = 2 * math.pi * f
    f2 = torch.where(wl > 8192.0, f * 8, f)
    smooth = (8192 / wl - 1) / 3
    f2 = torch.where((wl > 2048.0) & (wl < 8192.0), f2 / ((1 - smooth) / 8 + smooth), f2)
    return (1.0 / f2).to(DEV)


def exact(case, seed):
    inp = _inputs(case, seed)
    if case["kind"] in ("decode", "mixed"):
        k, v = _stored(case, inp["k"], inp["v"])
        return _attend(case, inp["q"], k, v, inp["qlens"], inp["kvl"])
    # the rotated queries; the angle is a 32-bit product, as the rotation defines it
    inv = _llama3_inv(case["d"])
    start = [0] * len(inp["kvl"]) if case["kind"] == "write" else inp["kvl"]
    pos = torch.cat([torch.arange(s, s + n) for s, n in zip(start, inp["qlens"])]).to(DEV)
    ang = (pos.float()[:, None] * inv).double()[:, None]

    def turn(x):
        half = x.shape[-1] // 2
        a, b = x[..., :half].double(), x[..., half:].double()
        return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], -1)

    q64 = turn(inp["q"])
    step, cache = case["kind"] == "step", case["cache"]
    kn, vn = _new_tokens(case, inp, seed) if step else (inp["k"], inp["v"])
    kn = turn(kn)
    if cache in ("f16", "bf16"):  # unquantized pages hold the rotated keys and the values themselves
        kp, vp = (inp["k"].double(), inp["v"].double()) if step else (kn, vn.double())
        pages = [_scatter(x, inp["slot"], inp["pool"], case["page"]) for x in (kp, vp)]
        if step:
            t = torch.from_numpy(inp["tables"]).to(DEV)
            n = torch.tensor(inp["kvl"], device=DEV)
            i = torch.arange(len(inp["kvl"]), device=DEV)
            for p, x in zip(pages, (kn, vn.double())):
                p[t[i, n // case["page"]].long(), n % case["page"]] = x
    else:
        pages = [None] * (4 if cache == "fp8" else 6)
    if not step:
        return [q64] + pages
    if cache == "fp8":  # the new token raises its page's scale for the earlier codes too: left out
        return [q64, None] + pages
    k, v = _stored(case, inp["k"], inp["v"])
    k2, v2 = _stored(case, kn.to(_dtype(case)), vn)
    at, ks, vs = 0, [], []
    for i, n in enumerate(inp["kvl"]):
        ks += [k[at:at + n], k2[i:i + 1]]
        vs += [v[at:at + n], v2[i:i + 1]]
        at += n
    out = _attend(case, q64.to(_dtype(case)), torch.cat(ks), torch.cat(vs), inp["qlens"], [n + 1 for n in inp["kvl"]])
    return [q64, out] + pages
