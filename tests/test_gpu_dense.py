"""The dense prefill kernel (q4kv_dense.hip: many tokens, 64 / 128 / 256 dims,
q8_0 and f16 caches) against the oracle where it can go wrong: column tiles
of 128 (tokens x query heads) with remainders, passes of 32 to 128 positions,
tiles split over workgroups and merged, a cache that ends before the tokens
do, unaligned queries, and values that are not finite in rows that only some
tokens see."""
import numpy as np
import pytest

import q4kv
from gpu_util import note, quantize_on_gpu
from synth import assert_attn_close, heads

pytestmark = pytest.mark.gpu


def _run(rt, q, gate, kc, vc, kind, n_kvh, base, max_kv, shift=0):
    """One decode_n call; shift moves q, gate and out by that many floats."""
    n_tok, n_head, hd = q.shape
    bufs = [rt.alloc(q.nbytes + 16) for _ in range(3)]
    for b, x in zip(bufs, (q, gate)):
        rt.h2d(b + 4 * shift, x)
    dq, dg, do = (b + 4 * shift for b in bufs)
    assert rt.lib.q4_hip_qsa_decode_n(dq, kc, vc, dg, do, n_head, n_kvh, hd, n_tok, base, max_kv,
                                      1.0 / np.sqrt(hd), kind)
    rt.sync()
    got = rt.download(do, q.nbytes, np.float32).reshape(q.shape)
    for b in bufs:
        rt.free(b)
    return got


def _inputs(seed, kind, n_head, n_kvh, hd, n_tok, ctx):
    rng = np.random.default_rng(seed)
    k, v = heads(rng, (ctx, n_kvh), hd=hd), heads(rng, (ctx, n_kvh), hd=hd)
    q = heads(rng, (n_tok, n_head), hd=hd)
    return k, v, q, rng.standard_normal(q.shape).astype(np.float32)


def _reaches_dense(hd, n_tok, n_head, n_kvh, kind, max_n):
    """q4kv_dense_takes for aligned caches: other calls run q4kv_rows.hip or
    the 256-dim decode kernels."""
    gqa = n_head // n_kvh
    if gqa > 16:
        return True
    hg = 2 if gqa > 8 else 1
    slots = n_tok * n_kvh * hg * (max_n - min(max_n, n_tok) // 2)
    tiles = -(-n_tok * gqa // 128) * n_kvh
    per_tile = n_tok * n_kvh * hg / tiles * min(1.0, tiles * 64 / 256)
    return (n_tok > 1 and slots > (280000 if hd == 256 else 160000)
            and per_tile > (1.5 if kind == q4kv.KV_F16 or hd == 64 else 2 if hd == 128 else 4))


# (kind, n_head, n_kvh, hd, n_tok, base, max_kv below base + n_tok, shift)
CASES = [
    (2, 24, 2, 256, 301, 640, 0, 0),    # 28.2 tiles in 4 splits
    (2, 24, 2, 256, 700, 0, 0, 0),      # causal from position 0: the last tiles split
    (1, 16, 2, 256, 130, 1999, 0, 0),   # f16
    (2, 8, 2, 256, 600, 700, 0, 1),     # 4 heads per KV head, unaligned queries
    (2, 20, 1, 256, 9, 33, 0, 0),       # more than 16 heads per KV head
    (2, 16, 2, 256, 280, 1000, 150, 0), # the cache ends before the tokens do
    (1, 32, 8, 128, 133, 195, 0, 0),    # 128 dims, 64 positions per pass
    (1, 16, 2, 128, 201, 3001, 0, 1),   # its tiles in 8 splits, unaligned queries
    (2, 32, 8, 128, 47, 2003, 0, 0),    # 12 splits, a tile of 60 columns
    (2, 40, 2, 128, 1, 5000, 0, 0),     # one token, 32 splits
    (2, 3, 1, 128, 705, 62, 40, 3),     # KV rows of 136 bytes, 6 splits
    (1, 24, 8, 64, 143, 127, 0, 0),     # 64 dims, 128 positions per pass
    (1, 24, 2, 64, 83, 2900, 0, 0),     # 12 splits
    (2, 36, 2, 64, 2, 0, 0, 0),         # the smallest prompt
    (2, 4, 4, 64, 129, 3000, 0, 0),     # one head per KV head, 12 splits
]


@pytest.mark.parametrize("kind,n_head,n_kvh,hd,n_tok,base,cut,shift", CASES)
def test_dense_prefill(rt, oracle, kind, n_head, n_kvh, hd, n_tok, base, cut, shift):
    note(f"dense kind={kind} heads={n_head}/{n_kvh} hd={hd} n_tok={n_tok} base={base} cut={cut}")
    ctx = base + n_tok
    assert _reaches_dense(hd, n_tok, n_head, n_kvh, kind, ctx - cut)
    k, v, q, gate = _inputs(31 * hd + n_tok, kind, n_head, n_kvh, hd, n_tok, ctx)
    kc, _ = quantize_on_gpu(rt, k, kind)
    vc, _ = quantize_on_gpu(rt, v, kind)
    got = _run(rt, q, gate, kc, vc, kind, n_kvh, base, ctx - cut, shift)
    want = oracle.attn(q, oracle.encode(k, kind), oracle.encode(v, kind), kind, n_head, n_kvh, hd,
                       n_tok, gate=gate, kv_base=base, max_kv=ctx - cut, threads=8)
    assert_attn_close(got, want, what=f"dense hd={hd} gqa={n_head // n_kvh}")
    for p in (kc, vc):
        rt.free(p)


@pytest.mark.parametrize("kind,hd", [(2, 128), (1, 128), (1, 64), (2, 256)])
def test_values_not_finite(rt, kind, hd):
    """inf / NaN in one V row: tokens that do not see it are bit-identical to
    the call without it, the others are not finite in exactly its dims (NaN, or
    inf where both parts of a weight have one sign)."""
    n_head, n_kvh, n_tok, base = 16, 2, 300, 1500
    note(f"dense V not finite kind={kind} hd={hd}")
    ctx, bad, kh = base + n_tok, base + 170, 1
    k, v, q, gate = _inputs(5 + hd, kind, n_head, n_kvh, hd, n_tok, ctx)
    kc, _ = quantize_on_gpu(rt, k, kind)
    vc, nb = quantize_on_gpu(rt, v, kind)
    clean = _run(rt, q, gate, kc, vc, kind, n_kvh, base, ctx)
    rows = rt.download(vc, nb).reshape(ctx, n_kvh, -1).copy()
    if kind == q4kv.KV_Q8:  # the scale of the row's second block
        rows[bad, kh].view(np.uint16)[17] = 0x7C00
        dims = np.arange(32, 64)
    else:
        rows[bad, kh].view(np.uint16)[[3, 40]] = (0x7E00, 0xFC00)
        dims = np.array([3, 40])
    rt.h2d(vc, rows)
    got = _run(rt, q, gate, kc, vc, kind, n_kvh, base, ctx)
    hit = np.zeros(q.shape, bool)
    hit[bad - base:, kh * n_head // n_kvh:, dims] = True
    assert not np.isfinite(got[hit]).any()
    assert np.array_equal(got[~hit], clean[~hit])
    for p in (kc, vc):
        rt.free(p)


@pytest.mark.parametrize("kind,hd", [(2, 256), (1, 256), (2, 128), (1, 64)])
def test_scores_not_finite(rt, kind, hd):
    """A NaN in one head's query: that head's row of that token is NaN, whether
    its tile is split or not, and no other one. A NaN in a K row: every token
    that sees the row is NaN in that KV head, no other one. (The others may
    round differently: a wave's columns move their maxima together.)"""
    n_head, n_kvh = 24, 2
    # the last half of the tiles is split (64 dims: all)
    n_tok, base = {256: (700, 0), 128: (1000, 0), 64: (300, 3000)}[hd]
    ctx = base + n_tok
    note(f"dense scores not finite kind={kind} hd={hd}")
    k, v, q, gate = _inputs(7 + hd, kind, n_head, n_kvh, hd, n_tok, ctx)
    kc, nb = quantize_on_gpu(rt, k, kind)
    vc, _ = quantize_on_gpu(rt, v, kind)
    clean = _run(rt, q, gate, kc, vc, kind, n_kvh, base, ctx)
    assert np.isfinite(clean).all()
    hit = np.zeros(q.shape, bool)
    qn = q.copy()
    for t in (0, 9, n_tok // 2, n_tok - 50, n_tok - 1):
        qn[t, (t * 5) % n_head, t % hd] = np.nan
        hit[t, (t * 5) % n_head] = True
    got = _run(rt, qn, gate, kc, vc, kind, n_kvh, base, ctx)
    assert np.isnan(got[hit]).all()
    assert_attn_close(got[~hit], clean[~hit])
    for row, kh in ((base + 40, 1), (ctx - 60, 0)):
        rows = rt.download(kc, nb).reshape(ctx, n_kvh, -1)
        bad = rows.copy()
        bad[row, kh].view(np.uint16)[17 if kind == q4kv.KV_Q8 else 40] = 0x7E00
        rt.h2d(kc, bad)
        got = _run(rt, q, gate, kc, vc, kind, n_kvh, base, ctx)
        rt.h2d(kc, rows)
        hit = np.zeros(q.shape, bool)
        hit[row - base:, kh * 12:kh * 12 + 12] = True
        assert np.isnan(got[hit]).all()
        assert_attn_close(got[~hit], clean[~hit])
    for p in (kc, vc):
        rt.free(p)


@pytest.mark.parametrize("hd", [256, 128])
def test_inf_beside_a_large_scale(rt, hd):
    """One pass holds a V row with an infinite scale and one with a scale past
    512 (V goes over to v * scale / 128 there): tokens that do not see the
    first are as without it, the others are not finite in its block only."""
    n_head, n_kvh, n_tok, base = 16, 2, 300, 1500
    note(f"dense inf beside a large scale hd={hd}")
    ctx, bad, kh = base + n_tok, base + 170, 1
    k, v, q, gate = _inputs(50 + hd, 2, n_head, n_kvh, hd, n_tok, ctx)
    v[bad + 2, kh, :32] *= np.float32(1e6)
    kc, _ = quantize_on_gpu(rt, k, 2)
    vc, nb = quantize_on_gpu(rt, v, 2)
    clean = _run(rt, q, gate, kc, vc, 2, n_kvh, base, ctx)
    assert np.isfinite(clean).all() and np.abs(clean).max() > 1e3
    rows = rt.download(vc, nb).reshape(ctx, n_kvh, -1).copy()
    rows[bad, kh].view(np.uint16)[17] = 0x7C00
    rt.h2d(vc, rows)
    got = _run(rt, q, gate, kc, vc, 2, n_kvh, base, ctx)
    hit = np.zeros(q.shape, bool)
    hit[bad - base:, kh * n_head // n_kvh:, 32:64] = True
    assert not np.isfinite(got[hit]).any()
    assert np.array_equal(got[~hit], clean[~hit])
    for p in (kc, vc):
        rt.free(p)
