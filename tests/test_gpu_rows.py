"""The 64- and 128-dim decode kernel (q4kv_rows.hip) against the oracle where
it can go wrong: lengths around its 16-entry passes, 64-entry rounds of four
waves and pieces, dense and listed items in one ragged batch, padding and
out-of-range entries, rows that are not listed and hold NaN, lists longer than
the launch was told, both head-group counts, and the fused-call step."""
import numpy as np
import pytest

import q4kv
from gpu_util import note
from synth import assert_attn_close, heads

pytestmark = pytest.mark.gpu

LENGTHS = (1, 15, 16, 17, 63, 65, 200, 900, 5000)


def _item(rng, oracle, kind, n_head, n_kvh, hd, n, listed):
    ctx = n + 40 if listed else n
    k, v = heads(rng, (ctx, n_kvh), hd=hd), heads(rng, (ctx, n_kvh), hd=hd)
    it = dict(ctx=ctx, n=n, sel=None, q=heads(rng, (1, n_head), hd=hd),
              gate=rng.standard_normal((n_head, hd)).astype(np.float32) if n % 2 else None)
    if listed:
        # n entries per KV head: positions 3.., a few padded or past the cache
        sel = np.stack([rng.permutation(ctx - 3)[:n] + 3 for _ in range(n_kvh)]).astype(np.int32)
        for row in sel:
            row[rng.random(n) < 0.1] = -1
            row[rng.random(n) < 0.02] = ctx + 5
        it["sel"] = sel
    kb, vb = oracle.encode(k, kind), oracle.encode(v, kind)
    it["want"] = oracle.attn(it["q"], kb, vb, kind, n_head, n_kvh, hd, 1,
                             gate=None if it["gate"] is None else it["gate"][None],
                             idx=it["sel"], width=n, tok_stride=n_kvh * n, kvh_stride=n,
                             kv_base=n - 1, max_kv=ctx, scale=1.0 / np.sqrt(hd), threads=8)
    if listed:
        # rows 0-2 are in no list: NaN (scales, or the values themselves)
        for b in (kb, vb):
            rows = b.view(np.uint8).reshape(ctx, n_kvh, -1)
            rows[:3].view(np.uint16)[..., ::17 if kind == q4kv.KV_Q8 else 1] = 0x7E00
    it["kc"], it["vc"] = kb, vb
    return it


@pytest.mark.parametrize("kind,n_head,n_kvh,hd", [
    (1, 32, 8, 128), (2, 32, 8, 128), (2, 24, 2, 128), (1, 24, 2, 128),
    (1, 16, 4, 64), (2, 16, 4, 64), (2, 64, 4, 64), (1, 3, 3, 64)])
def test_ragged_batch(rt, oracle, kind, n_head, n_kvh, hd):
    note(f"rows batch kind={kind} heads={n_head}/{n_kvh} hd={hd}")
    rng = np.random.default_rng(70 + kind + n_head + hd)
    items = [_item(rng, oracle, kind, n_head, n_kvh, hd, n, listed)
             for n in LENGTHS for listed in (False, True)]
    empty = _item(rng, oracle, kind, n_head, n_kvh, hd, 70, True)
    empty["sel"][:] = -1
    empty["want"][:] = 0.0
    items.append(empty)
    descs = (q4kv.SeqDesc * len(items))()
    before = set(rt._owned)
    for d, it in zip(descs, items):
        it["out"] = rt.alloc(it["q"].nbytes)
        d.kcache, d.vcache, d.q = rt.upload(it["kc"]), rt.upload(it["vc"]), rt.upload(it["q"])
        d.gate = None if it["gate"] is None else rt.upload(it["gate"])
        d.out = it["out"]
        d.idx = None if it["sel"] is None else rt.upload(it["sel"])
        d.n_sel, d.idx_kvh_stride, d.max_kv = it["n"], it["n"], it["ctx"]
    dd = rt.upload(np.frombuffer(bytes(descs), np.uint8))
    # told the true maximum (pieces and their merge), or too small a one (the
    # last piece takes the rest)
    for max_n in (5000, 64, 1):
        for it in items:
            rt.h2d(it["out"], np.full(it["q"].size, np.nan, np.float32))
        assert rt.lib.q4_hip_qsa_decode_batch(dd, len(items), n_head, n_kvh, hd,
                                              1.0 / np.sqrt(hd), kind, max_n)
        rt.sync()
        for it in items:
            got = rt.download(it["out"], it["q"].nbytes, np.float32).reshape(it["q"].shape)
            assert_attn_close(got, it["want"], what=f"n={it['n']} listed={it['sel'] is not None} "
                                                    f"max_n={max_n}")
    for p in [p for p in rt._owned if p not in before]:
        rt.free(p)


@pytest.mark.parametrize("kind,hd", [(1, 128), (2, 64)])
def test_step_equals_append_then_batch(rt, oracle, kind, hd):
    """q4_hip_qsa_step_batch: the appended row is attended, and the outputs
    equal the append and the batched decode called one after the other."""
    note(f"rows step kind={kind} hd={hd}")
    rng = np.random.default_rng(hd + kind)
    n_head, n_kvh, n = 16, 4, 333
    k, v = heads(rng, (n, n_kvh), hd=hd), heads(rng, (n, n_kvh), hd=hd)
    q = heads(rng, (1, n_head), hd=hd)
    kb, vb = oracle.encode(k, kind), oracle.encode(v, kind)
    row = kb.nbytes // n
    before = set(rt._owned)
    kz, vz = kb.copy(), vb.copy()
    for b in (kz, vz):
        b.view(np.uint8).reshape(n, -1)[-1] = 0
    kc, vc, out = rt.upload(kz), rt.upload(vz), rt.alloc(q.nbytes)
    step = q4kv.StepDesc(q4kv.SeqDesc(kc, vc, rt.upload(q), None, out, None, n, 0, n, 0),
                         rt.upload(k[-1]), rt.upload(v[-1]), n - 1)
    dd = rt.upload(np.frombuffer(bytes(step), np.uint8))
    args = (1, n_head, n_kvh, hd, 1.0 / np.sqrt(hd), kind, n)
    assert rt.lib.q4_hip_qsa_step_batch(dd, *args)
    rt.sync()
    assert np.array_equal(rt.download(kc, kb.nbytes)[-row:], kb.view(np.uint8).ravel()[-row:])
    got = rt.download(out, q.nbytes, np.float32).reshape(q.shape)
    want = oracle.attn(q, kb, vb, kind, n_head, n_kvh, hd, 1, kv_base=n - 1, max_kv=n)
    assert_attn_close(got, want, what="step")
    assert rt.lib.q4_hip_qsa_decode_batch(rt.upload(np.frombuffer(bytes(step.seq), np.uint8)), *args)
    rt.sync()
    assert np.array_equal(rt.download(out, q.nbytes, np.float32).reshape(q.shape), got)
    for p in [p for p in rt._owned if p not in before]:
        rt.free(p)


@pytest.mark.parametrize("kind,n_head,n_kvh,hd", [(1, 32, 8, 128), (2, 24, 2, 128), (2, 16, 4, 64)])
def test_weights_are_rounded(rt, oracle, kind, n_head, n_kvh, hd):
    """Equal V everywhere, so every output is that value whatever the weights:
    the sum of the weights' fp16 parts over the fp32 sum of the weights. Parts
    cut off after 21 bits (an error of 0 to 2^-21, one sign) lower the mean by
    7e-8 to 9e-8; rounded ones leave no mean but that of the fp32 sums, less
    than the half ulp 2^-24 of a single one (1.5e-8 at most seen)."""
    note(f"rows weights kind={kind} heads={n_head}/{n_kvh} hd={hd}")
    rng = np.random.default_rng(3 * hd + kind)
    n, before = 3000, set(rt._owned)
    k, v = heads(rng, (n, n_kvh), hd=hd), np.ones((n, n_kvh, hd), np.float32)
    q = rng.standard_normal((1, n_head, hd)).astype(np.float32) * np.float32(0.3)
    kc, vc = rt.upload(oracle.encode(k, kind)), rt.upload(oracle.encode(v, kind))
    value = 127.0 * float(np.float16(np.float32(1) / np.float32(127))) if kind == q4kv.KV_Q8 else 1.0
    out = rt.alloc(q.nbytes)
    sel = rt.upload(np.arange(n, dtype=np.int32))
    assert rt.lib.q4_hip_qsa_decode_idx_kv(rt.upload(q), kc, vc, None, out, sel, n, n, 0, n_head,
                                           n_kvh, hd, 1, n, 1.0 / np.sqrt(hd), kind)
    rt.sync()
    got = rt.download(out, q.nbytes, np.float32).astype(np.float64) / value - 1.0
    assert abs(got.mean()) <= 2.0 ** -24, got.mean()
    for p in [p for p in rt._owned if p not in before]:
        rt.free(p)


@pytest.mark.parametrize("kind,hd", [(1, 128), (2, 64)])
def test_scores_not_finite(rt, oracle, kind, hd):
    """A NaN in a head's query, or in a K row, reaches that head's (that KV
    head's) output whether the item is one piece or many."""
    note(f"rows scores not finite kind={kind} hd={hd}")
    rng = np.random.default_rng(hd)
    n_head, n_kvh, before = 16, 4, set(rt._owned)
    out = rt.alloc(n_head * hd * 4)
    for n in (60, 5000):
        k, v = heads(rng, (n, n_kvh), hd=hd), heads(rng, (n, n_kvh), hd=hd)
        q = heads(rng, (1, n_head), hd=hd)
        gate = rt.upload(np.zeros_like(q))
        kb, vc = oracle.encode(k, kind), rt.upload(oracle.encode(v, kind))
        qn, kn = q.copy(), kb.copy()
        qn[0, 5, 7] = np.nan
        kn.view(np.uint8).reshape(n, n_kvh, -1)[n // 3, 2].view(np.uint16)[17] = 0x7E00
        for qx, kx, hit in ((qn, kb, [5]), (q, kn, [8, 9, 10, 11])):
            assert rt.lib.q4_hip_qsa_decode(rt.upload(qx), rt.upload(kx), vc, gate, out, n_head,
                                            n_kvh, hd, n, n, 1.0 / np.sqrt(hd), kind)
            rt.sync()
            got = rt.download(out, q.nbytes, np.float32).reshape(n_head, hd)
            assert np.isnan(got[hit]).all(), n
            assert np.isfinite(np.delete(got, hit, 0)).all(), n
    for p in [p for p in rt._owned if p not in before]:
        rt.free(p)
