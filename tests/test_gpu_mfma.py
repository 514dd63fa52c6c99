"""MFMA attention over every cache type (unquantized fp16 / bf16, FP8, affine pages) vs the float64 oracle.

Bound of a result: half a unit in the last place of the 16-bit output (2^-11 / 2^-8 of the value, bf16
rounding 8 bits) plus the fp32 arithmetic: scores are fp32 sums of up to 256 products, |s| <= ~16, so a
probability is off by at most ~2^-18 of itself and an output by 2^-16 of the largest value it averages.
"""

import numpy as np
import pytest
import torch

from easymlx_amd import paged_attention
from easymlx_amd.caching import layout
from oracle import fp8
from oracle.paged_attention import paged_attention as oracle_attention

pytestmark = pytest.mark.gpu

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "fp8": torch.float16, "q4": torch.float16, "q8": torch.float16}


def batch(kind, qlens, kvl, hq, hkv, d, page, seed, invalid=(), gs=64):
    """Seeded inputs on the CPU: queries, stored caches (and scales), tables, and the exact cache values."""
    rng = np.random.default_rng(seed)
    pages = [-(-max(x, 1) // page) for x in kvl]
    nb = sum(pages) + 1
    tables = np.full((len(kvl), max(pages)), -1, np.int32)
    perm, at = rng.permutation(nb).astype(np.int32), 0
    for i, p in enumerate(pages):
        tables[i, :p] = perm[at:at + p]
        at += p
    for i, c in invalid:
        tables[i, c] = -1 if c % 2 else nb + 3
    q = torch.from_numpy(rng.standard_normal((sum(qlens), hq, d), dtype=np.float32)).to(DTYPES[kind])
    shape = (nb, page, hkv, d)
    scales = None
    if kind == "fp8":
        codes = [rng.integers(0, 256, size=shape).astype(np.uint8) & 0xF7 for _ in range(2)]  # |x| <= 240, no NaN code
        scales = [rng.uniform(0.003, 0.02, size=nb).astype(np.float32) for _ in range(2)]
        cache = [torch.from_numpy(c) for c in codes]
        exact = [fp8.e4m3_decode(c).astype(np.float64) * s[:, None, None, None].astype(np.float64)
                 for c, s in zip(codes, scales)]
    elif kind in ("q4", "q8"):
        bits = int(kind[1])
        cache, exact, scales = [], [], {"bits": bits, "group_size": gs}
        for name, pack in (("k", layout.key_pages_from_logical), ("v", lambda w: layout.value_pages_from_logical(w, bits))):
            codes = rng.integers(0, 1 << bits, size=shape)
            sc = (rng.uniform(0.5, 2.0, size=shape[:3] + (d // gs,)) * rng.choice([-1, 1], size=shape[:3] + (d // gs,))
                  * 6.0 / (1 << bits)).astype(np.float16)
            bi = (-sc.astype(np.float32) * (1 << (bits - 1)) + rng.standard_normal(sc.shape) * 0.3).astype(np.float16)
            exact.append(codes * np.repeat(sc.astype(np.float64), gs, -1) + np.repeat(bi.astype(np.float64), gs, -1))
            cache.append(torch.from_numpy(pack(layout._pack(codes, bits)).view(np.int32)))
            scales[name + "_scales"] = torch.from_numpy(layout.params_pages_from_logical(sc))
            scales[name + "_biases"] = torch.from_numpy(layout.params_pages_from_logical(bi))
    else:
        cache = [torch.from_numpy(rng.standard_normal(shape, dtype=np.float32) * 1.5).to(DTYPES[kind])
                 for _ in range(2)]
        exact = [c.double().numpy() for c in cache]
    return dict(q=q, cache=cache, scales=scales, exact=exact, tables=tables, kvl=np.asarray(kvl, np.int32),
                qsl=np.concatenate([[0], np.cumsum(qlens)]).astype(np.int32))


def run(b, dev, window=0, decode=True, out=None):
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    sc = b["scales"]
    if isinstance(sc, dict):
        kw = {k: x.to(dev) if isinstance(x, torch.Tensor) else x for k, x in sc.items()}
    else:
        kw = dict(k_scale=t(sc[0]), v_scale=t(sc[1])) if sc is not None else {}
    out = paged_attention(b["q"].to(dev), b["cache"][0].to(dev), b["cache"][1].to(dev), t(b["tables"]), t(b["kvl"]),
                          t(b["qsl"]), sliding_window=window or None, single_token_decode=decode, out=out, **kw)
    torch.cuda.synchronize()
    return out.double().cpu().numpy()


def expected(b, window=0):
    return oracle_attention(b["q"].double().numpy(), b["exact"][0], b["exact"][1], b["tables"], b["kvl"], b["qsl"],
                            sliding_window=window, compute_dtype=np.float64, out_dtype=np.float64)


def check(b, got, exp):
    ulp = 2.0 ** -8 if b["q"].dtype == torch.bfloat16 else 2.0 ** -11
    bound = ulp * np.abs(exp) + 2.0 ** -16 * np.abs(b["exact"][1]).max() + 2.0 ** -24
    err = np.abs(got - exp)
    assert np.isfinite(got).all()
    assert (err <= bound).all(), f"{int((err > bound).sum())} of {err.size}, worst {(err / bound).max():.2f} of the bound"


def affine_bound(b, exp):
    """prefill_affine rounds values and probabilities to fp16: 2^-11 of the largest value each, beside the output's."""
    return 2.0 ** -11 * np.abs(exp) + 2 * 2.0 ** -11 * np.abs(b["exact"][1]).max()


# item (128), wave (32) and quad (4) edges, and contexts cut between workgroups
CONTEXTS = [1, 3, 31, 32, 33, 127, 128, 129, 0, 300, 1000, 5]


@pytest.mark.parametrize("kind", ["f16", "bf16", "fp8"])
@pytest.mark.parametrize("d,page,hq,hkv", [(64, 16, 8, 2), (128, 16, 6, 2), (128, 24, 7, 1), (128, 8, 40, 2),
                                           (256, 64, 4, 4), (256, 32, 16, 1)])
def test_decode(cuda, kind, d, page, hq, hkv):
    print(f"[token-major decode {kind} d{d} page{page} {hq}/{hkv}]", flush=True)
    b = batch(kind, [1] * len(CONTEXTS), CONTEXTS, hq, hkv, d, page, seed=d + page + hq,
              invalid=[(5, 1), (9, 0), (10, 2)] if page < 64 else [])
    for window in (0, 1, 100):
        check(b, run(b, cuda, window), expected(b, window))


# shapes the 128-wide affine decode kernels do not take: other head sizes, GQA ratios that are not
# powers of two (or above 16), pages between theirs
@pytest.mark.parametrize("kind", ["q4", "q8"])
@pytest.mark.parametrize("d,page,hq,hkv,gs", [(64, 16, 8, 2, 64), (64, 128, 4, 4, 64), (128, 16, 6, 2, 64),
                                              (128, 32, 40, 2, 128), (128, 192, 7, 1, 64), (256, 64, 4, 4, 64),
                                              (256, 16, 16, 1, 128), (256, 128, 9, 3, 64)])
def test_decode_affine(cuda, kind, d, page, hq, hkv, gs):
    print(f"[affine decode {kind} d{d} page{page} {hq}/{hkv} g{gs}]", flush=True)
    b = batch(kind, [1] * len(CONTEXTS), CONTEXTS, hq, hkv, d, page, seed=d + page + hq, gs=gs,
              invalid=[(5, 1), (9, 0), (10, 2)] if page < 64 else [])
    for window in (0, 1, 100):
        check(b, run(b, cuda, window), expected(b, window))


@pytest.mark.parametrize("kind", ["f16", "fp8"])
def test_decode_one_long_row(cuda, kind):
    """One sequence cut over every workgroup: a merge of many pieces, twice on the same workspace."""
    print(f"[token-major long row {kind}]", flush=True)
    b = batch(kind, [1], [40_003], 4, 1, 128, 16, seed=3)
    exp = expected(b)
    first = run(b, cuda)
    check(b, first, exp)
    assert np.array_equal(first, run(b, cuda))


def test_decode_affine_stale_scales(cuda):
    """Scales of tokens past kv_len may hold anything; an infinite scale of a live token gives infinities."""
    print("[affine decode stale scales]", flush=True)
    b = batch("q8", [1, 1], [70, 41], 6, 2, 128, 16, seed=4)
    exp = expected(b)
    at = lambda s, p: (int(b["tables"][s, p // 16]), p % 16)  # noqa: E731
    blk, off = at(0, 75)
    for n in ("k_scales", "k_biases", "v_scales", "v_biases"):
        b["scales"][n][blk, :, :, off] = float("nan")
    blk, off = at(1, 40)
    b["scales"]["v_biases"][blk, 1, 0, off] = float("inf")  # kv head 1, dims 0 .. 63
    got = run(b, cuda)
    assert np.isposinf(got[1, 3:, :64]).all()
    got[1, 3:, :64] = exp[1, 3:, :64]
    check(b, got, exp)


def test_decode_short_contexts_whole_units(cuda):
    """More units than workgroups, contexts too short to cut: ranges start at unit starts."""
    print("[decode whole units]", flush=True)
    kvl = [int(x) for x in np.random.default_rng(1).integers(1, 400, size=150)]
    for kind in ("bf16", "q4"):
        b = batch(kind, [1] * 150, kvl, 6, 6, 64, 16, seed=12)
        check(b, run(b, cuda), expected(b))


def test_decode_units_just_past_the_workgroups(cuda):
    """520 and 528 equal long units over 512 workgroups are cut: as whole units a workgroup would hold two of them,
    twice an equal share, and the call take nearly twice the time of 512 units (1.5 times at most is asked for)."""
    print("[decode 65 and 66 long rows]", flush=True)
    one = batch("f16", [1] * 66, [4096] + [1] * 65, 16, 8, 64, 16, seed=14)
    one["tables"][:] = one["tables"][0]  # every sequence reads the same pages
    one["kvl"][:] = 4096
    exp, took = expected(one), {}
    for seqs in (64, 65, 66):
        b = dict(one, q=one["q"][:seqs], tables=one["tables"][:seqs], kvl=one["kvl"][:seqs], qsl=one["qsl"][:seqs + 1])
        check(b, run(b, cuda), exp[:seqs])
        q, k, v = b["q"].to(cuda), b["cache"][0].to(cuda), b["cache"][1].to(cuda)
        args = [torch.from_numpy(b[n]).to(cuda) for n in ("tables", "kvl", "qsl")]
        best = float("inf")
        for _ in range(5):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            for _ in range(20):
                paged_attention(q, k, v, *args, single_token_decode=True)
            t1.record()
            torch.cuda.synchronize()
            best = min(best, t0.elapsed_time(t1))
        took[seqs] = best
    assert took[65] < 1.5 * took[64] and took[66] < 1.5 * took[64], took


def test_decode_short_contexts_side_by_side(cuda):
    """200 workgroups with one short item each take about what 8 take: they share no slow memory (2.2 times as long
    where each read the dispatch packet, in host memory; 1.5 times at most is asked for)."""
    print("[decode 25 short rows]", flush=True)
    took = {}
    for seqs in (1, 25):
        b = batch("bf16", [1] * seqs, [12] * seqs, 32, 8, 64, 16, seed=15)
        check(b, run(b, cuda), expected(b))
        q, k, v = b["q"].to(cuda), b["cache"][0].to(cuda), b["cache"][1].to(cuda)
        args, out = [torch.from_numpy(b[n]).to(cuda) for n in ("tables", "kvl", "qsl")], torch.empty_like(q)
        side, g = torch.cuda.Stream(cuda), torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=side):
            for _ in range(40):  # (in a graph: the host takes longer than these kernels)
                paged_attention(q, k, v, *args, single_token_decode=True, out=out)
        took[seqs] = float("inf")
        for _ in range(5):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            g.replay()
            t1.record()
            torch.cuda.synchronize()
            took[seqs] = min(took[seqs], t0.elapsed_time(t1))
        check(b, out.double().cpu().numpy(), expected(b))
    assert took[25] < 1.5 * took[1], took


@pytest.mark.parametrize("kind", ["f16", "bf16"])
def test_decode_infinities(cuda, kind):
    """An infinity or NaN outside the visible keys leaves a row as it is; a visible infinity stays one."""
    print(f"[token-major infinities {kind}]", flush=True)
    kvl, window = [200, 200, 70], 64
    b = batch(kind, [1] * 3, kvl, 4, 2, 128, 16, seed=8)
    exp = expected(b, window)
    v = b["cache"][1]
    at = lambda s, p: (int(b["tables"][s, p // 16]), p % 16)  # noqa: E731
    v[at(0, 130)][0, 7] = float("inf")   # before the window, in a step the kernel reads
    v[at(2, 75)][1, 9] = float("nan")    # stale, past kv_len in the last page
    v[at(1, 190)][1, 3] = float("inf")   # visible to sequence 1, kv head 1
    got = run(b, cuda, window)
    assert np.isposinf(got[1, 2:, 3]).all()
    got[1, 2:, 3] = exp[1, 2:, 3]
    check(b, got, exp)


@pytest.mark.parametrize("kind,d,page", [("f16", 64, 16), ("bf16", 128, 8), ("f16", 256, 32), ("q4", 64, 16),
                                          ("q8", 256, 64)])
def test_decode_infinities_in_cut_rows(cuda, kind, d, page):
    """Rows cut over many workgroups: an infinity stays one wherever it lies, a page of NaN keys gives zeros (the sum
    of the probabilities is no number), the other rows and dims stay as they are; in about the time of finite rows."""
    print(f"[decode infinities, cut rows {kind} d{d}]", flush=True)
    kvl = [3000, 3000, 3000, 70]
    b = batch(kind, [1] * 4, kvl, 4, 2, d, page, seed=18)
    exp = expected(b)

    def timed():
        got, best = run(b, cuda), float("inf")
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)  # noqa: E731
        sc = b["scales"] or {}
        kw = {n: x.to(cuda) if isinstance(x, torch.Tensor) else x for n, x in sc.items()}
        args = [b["q"].to(cuda), b["cache"][0].to(cuda), b["cache"][1].to(cuda), t(b["tables"]), t(b["kvl"]), t(b["qsl"])]
        for _ in range(5):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            for _ in range(10):
                paged_attention(*args, single_token_decode=True, **kw)
            t1.record()
            torch.cuda.synchronize()
            best = min(best, t0.elapsed_time(t1) * 100)
        return got, best

    finite, us = timed()
    check(b, finite, exp)
    at = lambda s, p: (int(b["tables"][s, p // page]), p % page)  # noqa: E731
    dims = slice(9, 10)
    if kind in ("q4", "q8"):
        dims = slice(0, 64)
        blk, off = at(0, 1500)
        b["scales"]["v_biases"][blk, 1, 0, off] = float("inf")
        blk, off = at(1, 0)
        b["scales"]["v_biases"][blk, 1, 0, off] = float("inf")
        b["scales"]["k_biases"][at(2, 1000)[0], 0, 0, :] = float("nan")
    else:
        b["cache"][1][at(0, 1500)][1, 9] = float("inf")
        b["cache"][1][at(1, 0)][1, 9] = float("inf")
        b["cache"][0][at(2, 1000)[0], :, 0, 3] = float("nan")
    got, us2 = timed()
    assert np.isposinf(got[:2, 2:, dims]).all() and (got[2, :2] == 0).all()
    got[:2, 2:, dims], got[2, :2] = exp[:2, 2:, dims], exp[2, :2]
    check(b, got, exp)
    assert us2 < 8 * us + 50, (us, us2)


@pytest.mark.parametrize("kind", ["f16", "fp8", "q4", "q8"])
@pytest.mark.parametrize("d,hq,hkv", [(64, 128, 1), (64, 130, 2), (128, 72, 1), (256, 64, 1), (64, 4, 4)])
def test_item_edges_and_many_heads(cuda, kind, d, hq, hkv):
    """Contexts at the item edges of 4-bit pages (64 tokens a wave, 256 an item), up to 128 query heads per kv head
    (one query token a tile, eight head groups in the decode)."""
    print(f"[item edges {kind} d{d} {hq}/{hkv}]", flush=True)
    kvl = [63, 64, 65, 255, 256, 257, 511, 513]
    b = batch(kind, [1] * len(kvl), kvl, hq, hkv, d, 16, seed=d + hq)
    check(b, run(b, cuda), expected(b))
    lens = [(1, 257), (3, 65), (66, 256), (1, 1), (2, 64)]
    b = batch(kind, [q for q, _ in lens], [k for _, k in lens], hq, hkv, d, 16, seed=d + hq)
    check(b, run(b, cuda, decode=False), expected(b))


@pytest.mark.parametrize("kind", ["f16", "bf16", "fp8", "q4", "q8"])
@pytest.mark.parametrize("d,page,hq,hkv", [(64, 16, 14, 2), (128, 24, 6, 2), (128, 8, 40, 2), (256, 64, 4, 4)])
@pytest.mark.parametrize("longest", [32, 33, 64, 65])
def test_decode_contexts_of_one_wave(cuda, kind, d, page, hq, hkv, longest):
    """Contexts that one wave's tokens hold (32; 64 over 4-bit pages) go a unit to a wave; one longer, none does."""
    if kind in ("q4", "q8") and page in (8, 24):
        page = 16
    print(f"[decode one wave {kind} d{d} page{page} {hq}/{hkv} up to {longest}]", flush=True)
    kvl = [longest] + [int(x) for x in np.random.default_rng(longest).integers(0, 33, size=150)]
    b = batch(kind, [1] * len(kvl), kvl, hq, hkv, d, page, seed=d + longest, invalid=[(3, 0), (9, 1)] if page < 32 else [])
    for window in (0, 7):
        check(b, run(b, cuda, window), expected(b, window))
    if kind in ("f16", "bf16"):
        s = max(range(1, len(kvl)), key=lambda i: kvl[i] % page and kvl[i])
        exp, blk = expected(b), int(b["tables"][s, (kvl[s] - 1) // page])
        b["cache"][1][blk, (kvl[s] - 1) % page, 0, 5] = float("inf")
        if kvl[s] % page:
            b["cache"][0][blk, kvl[s] % page:] = float("nan")  # stale
        got, hg = run(b, cuda), hq // hkv
        assert np.isposinf(got[s, :hg, 5]).all()
        got[s, :hg, 5] = exp[s, :hg, 5]
        check(b, got, exp)


# chunks around the tile and step edges, over cached prefixes, beside single-token and empty rows
RAGGED = [(33, 40), (1, 129), (2, 2), (130, 700), (1, 1), (0, 5), (65, 65), (7, 3), (1, 600), (5, 0), (64, 1300)]


@pytest.mark.parametrize("kind", ["f16", "bf16", "fp8"])
@pytest.mark.parametrize("d,page,hq,hkv", [(64, 16, 8, 2), (128, 16, 6, 2), (128, 24, 7, 1), (128, 8, 40, 2),
                                           (128, 128, 4, 4), (256, 64, 4, 4), (256, 32, 16, 1)])
def test_ragged(cuda, kind, d, page, hq, hkv):
    if kind == "fp8" and page == 128:
        pytest.skip("prefill_affine_d128's shape (tests/test_gpu_fp8.py)")
    print(f"[token-major ragged {kind} d{d} page{page} {hq}/{hkv}]", flush=True)
    b = batch(kind, [q for q, _ in RAGGED], [k for _, k in RAGGED], hq, hkv, d, page, seed=d + page + hq,
              invalid=[(3, 1), (3, 2), (8, 0), (10, 3)] if page < 64 else [])
    for window in (0, 50):
        check(b, run(b, cuda, window, decode=False), expected(b, window))


@pytest.mark.parametrize("kind", ["q4", "q8"])
@pytest.mark.parametrize("d,page,hq,hkv,gs", [(64, 16, 8, 2, 64), (64, 128, 4, 4, 64), (128, 16, 6, 2, 64),
                                              (128, 32, 40, 2, 128), (128, 192, 7, 1, 64), (256, 64, 4, 4, 64),
                                              (256, 16, 16, 1, 128), (256, 128, 9, 3, 64)])
def test_ragged_affine(cuda, kind, d, page, hq, hkv, gs):
    print(f"[affine ragged {kind} d{d} page{page} {hq}/{hkv} g{gs}]", flush=True)
    b = batch(kind, [q for q, _ in RAGGED], [k for _, k in RAGGED], hq, hkv, d, page, seed=d + page + hq, gs=gs,
              invalid=[(3, 1), (3, 2), (8, 0), (10, 3)] if page < 64 else [])
    for window in (0, 50):
        check(b, run(b, cuda, window, decode=False), expected(b, window))


def test_ragged_affine_stale_scales(cuda):
    """Scales past a sequence's last key may hold anything."""
    print("[affine ragged stale scales]", flush=True)
    b = batch("q4", [40, 1], [60, 35], 6, 2, 64, 32, seed=6)
    exp = expected(b)
    for s_, p in ((0, 61), (1, 36)):
        for n in ("k_scales", "k_biases", "v_scales", "v_biases"):
            b["scales"][n][int(b["tables"][s_, p // 32]), :, :, p % 32] = float("nan")
    check(b, run(b, cuda, decode=False), exp)


@pytest.mark.parametrize("kind", ["f16", "bf16", "fp8", "q4"])
@pytest.mark.parametrize("pad", [(0, 1), (3, 0), (5, 300)], ids=str)
@pytest.mark.parametrize("seqs", [len(RAGGED), 70])
def test_ragged_rows_of_no_sequence(cuda, kind, pad, seqs):
    """Rows before query_start_loc[0] and past its last entry (a padded call) are zeros, the others as without."""
    print(f"[ragged padded {kind} {pad} {seqs} sequences]", flush=True)
    lens = (RAGGED * 7)[:seqs] if seqs > 64 else RAGGED
    qlens = [min(q, 9) for q, _ in lens] if seqs > 64 else [q for q, _ in lens]
    b = batch(kind, qlens, [min(k, 90) if seqs > 64 else k for _, k in lens], 6, 2, 128, 16, seed=21)
    b["q"] = torch.cat([torch.ones_like(b["q"][:1]).expand(pad[0], -1, -1), b["q"],
                        torch.ones_like(b["q"][:1]).expand(pad[1], -1, -1)])
    b["qsl"] = b["qsl"] + np.int32(pad[0])
    out = torch.full_like(b["q"], 7.0).to(cuda)
    check(b, run(b, cuda, decode=False, out=out), expected(b))


@pytest.mark.parametrize("kind", ["bf16", "q8"])
@pytest.mark.parametrize("keep", [1, 34, 100, 199])  # the 34th row is a single-token sequence's, cut inside a chunk
def test_ragged_query_start_loc_past_the_rows(cuda, kind, keep):
    """query_start_loc may run past the rows given: those given are as in the whole call, nothing else is touched."""
    print(f"[ragged {keep} rows of {sum(q for q, _ in RAGGED)} {kind}]", flush=True)
    b = batch(kind, [q for q, _ in RAGGED], [k for _, k in RAGGED], 6, 2, 128, 16, seed=22)
    exp = expected(b)[:keep]
    b["q"] = b["q"][:keep]
    check(b, run(b, cuda, decode=False), exp)


def test_ragged_without_workspace(cuda):
    """The C entry point with no workspace: single-token rows go as query tiles, no tile is cut."""
    from easymlx_amd import _native

    print("[token-major ragged, no workspace]", flush=True)
    b = batch("f16", [q for q, _ in RAGGED], [k for _, k in RAGGED], 4, 2, 128, 16, seed=5)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)  # noqa: E731
    q, k, v = b["q"].to(cuda), b["cache"][0].to(cuda), b["cache"][1].to(cuda)
    bt, kvl, qsl = t(b["tables"]), t(b["kvl"]), t(b["qsl"])
    out = torch.full_like(q, 7.0)
    _native.check(_native.load().emx_paged_attention_dense(
        q.data_ptr(), q.shape[0], 4, 128, _native.DTYPE_F16, k.data_ptr(), v.data_ptr(), k.shape[0], 16, 2,
        bt.data_ptr(), bt.shape[0], bt.shape[1], kvl.data_ptr(), qsl.data_ptr(), 1 / np.sqrt(128), 0, 0, None, 0,
        out.data_ptr(), _native.stream_ptr(cuda)))
    torch.cuda.synchronize()
    check(b, out.double().cpu().numpy(), expected(b))


@pytest.mark.parametrize("kind,page,seqs,qlen,ctx,hq,hkv", [
    ("f16", 16, 1, 1290, 1290, 64, 1), ("bf16", 16, 2, 645, 1300, 64, 1),  # about 645 tiles: in two parts
    ("f16", 16, 3, 560, 700, 64, 1),                                      # about 840: uncut
    ("q4", 128, 4, 190, 800, 128, 8), ("q4", 128, 4, 215, 800, 128, 8)])  # the affine kernel: cut, uncut
def test_ragged_many_tiles(cuda, kind, page, seqs, qlen, ctx, hq, hkv):
    """Tile counts on both sides of the lines at which fewer parts are cut, tiles longer than a part."""
    print(f"[ragged {seqs}x{qlen}/{ctx} {kind} {hq}/{hkv}]", flush=True)
    d = 128 if kind == "q4" else 64
    b = batch(kind, [qlen] * seqs + [1], [ctx] * seqs + [77], hq, hkv, d, page, seed=qlen)
    got, exp = run(b, cuda, decode=False), expected(b)
    if kind != "q4":
        check(b, got, exp)
        return
    assert (np.abs(got - exp) <= affine_bound(b, exp)).all()


@pytest.mark.parametrize("kind,page,seqs,qlen,ctx,hq,hkv,rows", [
    ("f16", 16, 1, 150, 1600, 64, 1, 3),                                    # 75 tiles: three parts
    ("f16", 16, 1, 400, 1500, 64, 1, 1), ("bf16", 16, 2, 300, 700, 64, 1, 1),  # 200 and 300: two, in two and three places
    ("f16", 16, 2, 700, 2700, 64, 1, 1), ("q4", 128, 2, 340, 2700, 128, 8, 1),  # 700, 688, long contexts: two
    ("f16", 16, 3, 150, 1600, 64, 1, 80), ("q4", 128, 3, 150, 1600, 128, 8, 80)])  # the workgroup's scan, cut
def test_ragged_parts(cuda, kind, page, seqs, qlen, ctx, hq, hkv, rows):
    """Each number of parts and places a tile can have, beside single-token rows (80: more than 64 sequences)."""
    print(f"[ragged parts {seqs}x{qlen}/{ctx} beside {rows} {kind} {hq}/{hkv}]", flush=True)
    d = 128 if kind == "q4" else 64
    ctxs = [ctx - 37 * i for i in range(seqs)]
    b = batch(kind, [qlen] * seqs + [1] * rows, ctxs + [77] * rows, hq, hkv, d, page, seed=qlen + rows)
    exp = expected(b)
    for _ in range(2):  # the arrival counters are back at zero
        got = run(b, cuda, decode=False)
        if kind == "q4":
            assert (np.abs(got - exp) <= affine_bound(b, exp)).all()
        else:
            check(b, got, exp)


@pytest.mark.parametrize("kind,page,hq", [("f16", 16, 6), ("q4", 128, 8)])  # prefill_mfma, prefill_affine
@pytest.mark.parametrize("seqs", [15, 16, 17, 33, 63, 64, 65, 130])
def test_ragged_sequence_counts(cuda, kind, page, hq, seqs):
    """Tiles found by a wave's scan (rows of 16 lanes, up to 64 sequences) and by the workgroup's."""
    print(f"[ragged {seqs} sequences {kind}]", flush=True)
    rng = np.random.default_rng(seqs)
    qlens = [int(x) for x in rng.choice([0, 1, 2, 31, 64, 65], size=seqs)]
    qlens[-1] = 40  # the last lane holds a tile
    b = batch(kind, qlens, [n + int(x) for n, x in zip(qlens, rng.integers(0, 60, size=seqs))], hq, 2, 128, page,
              seed=seqs)
    got, exp = run(b, cuda, decode=False), expected(b)
    if kind == "f16":
        check(b, got, exp)
    else:
        assert (np.abs(got - exp) <= affine_bound(b, exp)).all()


def test_ragged_captured(cuda):
    """A ragged call over unquantized pages in a graph, after a smaller call on the stream: each replay as eager."""
    print("[token-major ragged, captured]", flush=True)
    small = batch("f16", [1, 1], [20, 30], 4, 2, 128, 16, seed=2)
    b = batch("f16", [q for q, _ in RAGGED], [k for _, k in RAGGED], 4, 2, 128, 16, seed=5)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)  # noqa: E731
    q, k, v = b["q"].to(cuda), b["cache"][0].to(cuda), b["cache"][1].to(cuda)
    args, out = [t(b[n]) for n in ("tables", "kvl", "qsl")], torch.empty_like(q)
    exp = expected(b)
    side = torch.cuda.Stream(cuda)
    with torch.cuda.stream(side):
        run(small, cuda)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        paged_attention(q, k, v, *args, single_token_decode=False, out=out)
    for _ in range(3):
        out.fill_(7.0)
        g.replay()
        torch.cuda.synchronize()
        check(b, out.double().cpu().numpy(), exp)
        with torch.cuda.stream(side):  # eager work on the stream of the capture
            check(b, run(b, cuda, decode=False), exp)


@pytest.mark.parametrize("kind,page,decode", [("f16", 16, True), ("q4", 128, True), ("q4", 16, False),
                                              ("q4", 128, False), ("fp8", 16, False), ("bf16", 16, False)])
def test_captured_past_the_streams_buffer(cuda, kind, page, decode):
    """Two captures that need more than the stream's buffer: eager work before any replay, the second replayed first."""
    print(f"[captured past the buffer {kind} p{page} {'decode' if decode else 'ragged'}]", flush=True)
    small = batch(kind, [1], [20], 4, 2, 128, page, seed=2)
    lens = [(1, k) for k in [700, 3, 129, 0, 2000] * 8] if decode else RAGGED
    b = batch(kind, [q for q, _ in lens], [k for _, k in lens], 4, 2, 128, page, seed=5)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)  # noqa: E731
    q, k, v = b["q"].to(cuda), b["cache"][0].to(cuda), b["cache"][1].to(cuda)
    sc = b["scales"]
    if isinstance(sc, dict):
        kw = {n: x.to(cuda) if isinstance(x, torch.Tensor) else x for n, x in sc.items()}
    else:
        kw = dict(k_scale=t(sc[0]), v_scale=t(sc[1])) if sc is not None else {}
    args, outs = [t(b[n]) for n in ("tables", "kvl", "qsl")], [torch.empty_like(q) for _ in range(2)]
    exp = expected(b)

    def right(out):
        got = out.double().cpu().numpy() if isinstance(out, torch.Tensor) else out
        if kind == "q4" and page == 128:
            assert (np.abs(got - exp) <= affine_bound(b, exp)).all()
        else:
            check(b, got, exp)

    side = torch.cuda.Stream(cuda)
    with torch.cuda.stream(side):
        run(small, cuda)
    torch.cuda.synchronize()
    graphs = []
    for out in outs:
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], stream=side):
            for _ in range(2):  # two layers share the capture's buffer
                paged_attention(q, k, v, *args, single_token_decode=decode, out=out, **kw)
    with torch.cuda.stream(side):
        run(small, cuda, decode=decode)
        right(run(b, cuda, decode=decode))
    for _ in range(3):
        for g, out in zip(graphs[::-1], outs[::-1]):
            out.fill_(7.0)
            g.replay()
            torch.cuda.synchronize()
            right(out)
        with torch.cuda.stream(side):
            right(run(b, cuda, decode=decode))


def test_ragged_infinities(cuda):
    """A value a row does not see (a later token of the prompt, a stale one) leaves it as it is."""
    print("[token-major ragged infinities]", flush=True)
    b = batch("bf16", [40, 1], [60, 30], 4, 2, 128, 16, seed=9)
    exp = expected(b)
    at = lambda s, p: (int(b["tables"][s, p // 16]), p % 16)  # noqa: E731
    b["cache"][1][at(0, 55)][0, 7] = float("inf")  # query rows 35 .. 39 see it, kv head 0
    b["cache"][1][at(1, 31)][1, 3] = float("nan")
    got = run(b, cuda, decode=False)
    assert np.isposinf(got[35:40, :2, 7]).all()
    got[35:40, :2, 7] = exp[35:40, :2, 7]
    check(b, got, exp)
