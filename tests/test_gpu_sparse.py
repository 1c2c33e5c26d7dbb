"""The listed-prefill kernel (q4kv_sparse.hip) against the oracle where it can
go wrong: both head packings, splits and the single split with the band apart,
lists whose length is not whole passes, padding anywhere (also whole passes
and whole lists of it), positions past the cache, rows that are in no list and
hold NaN, shared and per-KV-head lists."""
import numpy as np
import pytest

import q4kv
from gpu_util import note, quantize_on_gpu
from synth import assert_attn_close, heads

pytestmark = pytest.mark.gpu


def _lists(rng, n, width, ctx, run):
    """[n][width] distinct positions >= 3; some rows end in a run of `run`
    consecutive ones (a causal window), some have padding."""
    sel = np.empty((n, width), np.int32)
    for t in range(n):
        row = np.sort(rng.permutation(ctx - 3 - run)[:width]) + 3
        if run and t % 7 != 3:
            row[-run:] = ctx - run - (n - 1 - t) // 2 % 64 + np.arange(run)
        sel[t] = row
        kind = t % 5
        if kind == 1:
            sel[t, rng.random(width) < 0.2] = -1
        elif kind == 2:
            sel[t, 40:120] = -1  # whole passes
        elif kind == 3:
            sel[t, rng.random(width) < 0.05] = ctx + 9
    sel[n // 2] = -1
    return sel


# (n_head, n_kvh, n_tok, width, per KV head, run): splits, one split, the
# band; 9 to 16 and 1 to 8 heads per KV head
@pytest.mark.parametrize("n_head,n_kvh,n_tok,width,per_kvh,run", [
    (24, 2, 16, 2051, False, 0),     # 8 splits of 8 passes or more
    (24, 2, 17, 2051, False, 0),     # 7 splits, a token's KV heads not on one XCD
    (24, 2, 24, 2051, False, 90),    # 5 splits, grouped again
    (16, 1, 41, 2051, False, 0),     # 6 splits
    (24, 2, 130, 300, False, 70),    # one split
    (18, 2, 140, 257, True, 0),
    (32, 2, 1030, 261, False, 90),   # many tokens, short lists: the band stays in them
    (24, 2, 1026, 256, True, 256),   # lists that are all band
    (32, 2, 1030, 1537, False, 500), # the band apart, 16 heads
    (18, 2, 1025, 1600, True, 90),
    (10, 1, 2049, 1539, False, 90),  # an odd number of items
    (8, 1, 1601, 259, False, 70),    # the band and the slab kernel, odd
    (16, 2, 200, 259, False, 0),     # packed, 8 heads
    (4, 2, 220, 300, True, 64),      # packed, 2 heads
    (3, 3, 128, 290, False, 0),      # one head per KV head
])
def test_listed_prefill(rt, oracle, n_head, n_kvh, n_tok, width, per_kvh, run):
    note(f"sparse heads={n_head}/{n_kvh} n_tok={n_tok} width={width} per_kvh={per_kvh} run={run}")
    rng = np.random.default_rng(n_head * 1000 + n_tok + width)
    ctx, hd = 2600 if width > 1000 else 1400, 256
    k, v = heads(rng, (ctx, n_kvh)), heads(rng, (ctx, n_kvh))
    q = heads(rng, (n_tok, n_head))
    gate = rng.standard_normal(q.shape).astype(np.float32)
    kc, nb = quantize_on_gpu(rt, k, q4kv.KV_Q8)
    vc, _ = quantize_on_gpu(rt, v, q4kv.KV_Q8)
    kb, vb = oracle.encode(k, q4kv.KV_Q8), oracle.encode(v, q4kv.KV_Q8)
    nl = n_kvh if per_kvh else 1
    sel = np.stack([_lists(rng, n_tok, width, ctx, run) for _ in range(nl)], 1)
    want = oracle.attn(q, kb, vb, q4kv.KV_Q8, n_head, n_kvh, hd, n_tok, gate=gate, idx=sel.ravel(),
                       width=width, tok_stride=nl * width, kvh_stride=width if per_kvh else 0,
                       max_kv=ctx, threads=8)
    for c in (kc, vc):  # rows 0-2 are in no list
        rows = rt.download(c, nb).reshape(ctx, -1).copy()
        rows[:3].view(np.uint16)[:, ::17] = 0x7E00
        rt.h2d(c, rows)
    dq, dg, di = rt.upload(q), rt.upload(gate), rt.upload(sel)
    do = rt.alloc(q.nbytes)
    rt.h2d(do, np.full(q.size, np.nan, np.float32))
    assert rt.lib.q4_hip_qsa_decode_idx_kv(dq, kc, vc, dg, do, di, width, nl * width,
                                           width if per_kvh else 0, n_head, n_kvh, hd, n_tok, ctx,
                                           1.0 / 16, q4kv.KV_Q8)
    rt.sync()
    assert_attn_close(rt.download(do, q.nbytes, np.float32).reshape(q.shape), want,
                      what=f"listed prefill gqa={n_head // n_kvh}")
    for p in (kc, vc, dq, dg, di, do):
        rt.free(p)


@pytest.mark.parametrize("n_head,n_tok,width", [(24, 1030, 1537), (16, 1030, 261)])
def test_scores_not_finite(rt, n_head, n_tok, width):
    """A NaN in a K row reaches the tokens that list it, in the shared window
    (attended apart) as well as before it; both kernels that take the rest."""
    note(f"sparse scores not finite heads={n_head} n_tok={n_tok}")
    n_kvh, hd, run = 2, 256, 90
    rng = np.random.default_rng(n_head)
    ctx = 2600 if width > 1000 else 1400
    sel = _lists(rng, n_tok, width, ctx, run)
    q = heads(rng, (n_tok, n_head))
    k, v = heads(rng, (ctx, n_kvh)), heads(rng, (ctx, n_kvh))
    kc, nb = quantize_on_gpu(rt, k, q4kv.KV_Q8)
    vc, _ = quantize_on_gpu(rt, v, q4kv.KV_Q8)
    dq, di, do = rt.upload(q), rt.upload(sel), rt.alloc(q.nbytes)

    def run_once():
        assert rt.lib.q4_hip_qsa_decode_idx_kv(dq, kc, vc, None, do, di, width, width, 0, n_head,
                                               n_kvh, hd, n_tok, ctx, 1.0 / 16, q4kv.KV_Q8)
        rt.sync()
        return rt.download(do, q.nbytes, np.float32).reshape(q.shape)

    assert np.isfinite(run_once()).all()
    rows = rt.download(kc, nb).reshape(ctx, n_kvh, -1)
    for row in (ctx - 70, 100):  # a window row, a row before the windows
        bad = rows.copy()
        bad[row, 1].view(np.uint16)[17] = 0x7E00
        rt.h2d(kc, bad)
        got = run_once()
        hit = np.zeros(q.shape, bool)
        hit[(sel == row).any(1), n_head // 2:] = True
        assert hit.any() and np.isnan(got[hit]).all()
        assert np.isfinite(got[~hit]).all()
    for p in (kc, vc, dq, di, do):
        rt.free(p)


@pytest.mark.parametrize("n_head,n_tok,width", [(24, 40, 2051), (24, 260, 2051), (16, 210, 2051),
                                                (24, 1030, 700)])
def test_mostly_padding(rt, oracle, n_head, n_tok, width):
    """Lists of a prompt's first tokens (t + 1 positions, then padding) and
    lists with a few entries in passes far apart: passes without an entry are
    passed over, at the start, in between and at the end of a wave's share."""
    note(f"sparse padding heads={n_head} n_tok={n_tok} width={width}")
    n_kvh, hd, ctx = 2, 256, 1400
    rng = np.random.default_rng(n_head + n_tok)
    sel = np.full((n_tok, width), -1, np.int32)
    for t in range(n_tok):
        if t % 3 == 2:  # 1 to 12 entries anywhere
            at = rng.choice(width, 1 + t % 12, replace=False)
            sel[t, at] = rng.choice(ctx, at.size, replace=False)
        elif t % 3 == 1:  # one entry alone: the list's first, last, any pass
            sel[t, (0, width - 1, 32 * (t % (width // 32)))[t // 3 % 3]] = t
        else:
            n = min(t + 1, width, ctx)
            sel[t, :n] = np.arange(n)
    k, v = heads(rng, (ctx, n_kvh)), heads(rng, (ctx, n_kvh))
    q = heads(rng, (n_tok, n_head))
    kc, _ = quantize_on_gpu(rt, k, q4kv.KV_Q8)
    vc, _ = quantize_on_gpu(rt, v, q4kv.KV_Q8)
    want = oracle.attn(q, oracle.encode(k, 2), oracle.encode(v, 2), q4kv.KV_Q8, n_head, n_kvh, hd,
                       n_tok, idx=sel.ravel(), width=width, tok_stride=width, kvh_stride=0,
                       max_kv=ctx, threads=8)
    dq, di, do = rt.upload(q), rt.upload(sel), rt.alloc(q.nbytes)
    rt.h2d(do, np.full(q.size, np.nan, np.float32))
    assert rt.lib.q4_hip_qsa_decode_idx_kv(dq, kc, vc, None, do, di, width, width, 0, n_head,
                                           n_kvh, hd, n_tok, ctx, 1.0 / 16, q4kv.KV_Q8)
    rt.sync()
    assert_attn_close(rt.download(do, q.nbytes, np.float32).reshape(q.shape), want,
                      what=f"padding gqa={n_head // n_kvh}")
    for p in (kc, vc, dq, di, do):
        rt.free(p)
