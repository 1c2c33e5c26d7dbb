"""Performance cases of the QSA KV-cache library (libq4kv.so) on one GPU.

What an engine does with the library, through the C ABI's Python binding:

  eager          one token, short context, no indexer: the two one-row cache
                 writes and the dense decode of one layer (the smallest call)
  token          one decode token through `layers` layers in the order a
                 layer runs: device position, held append, fused decode
                 indexer, top-k, attention over the selected positions
  step           one decode step of many independent items (sequences, or the
                 layers of one sequence) in one call, appends included; with
                 or without the Q/K preparation in the same launch
  prefill        the tokens of one prompt slice or chunk: cache write, then
                 causal attention, dense or over per-token selections
  index_prefill  the indexer of a prompt slice: raw key store, block pooling,
                 scores, top-k selection per token
  index_batch    the decode indexer of many independent items in one call

Values: K, V and queries are N(0, 1) with four outlier channels x8 per head,
gates N(0, 1); selections are 2051 wide: three sinks, the 512 most recent
positions and 1536 earlier ones, or 512 blocks of four positions as the
indexer emits them. Sizes: 24 or 16 query heads over 2 KV heads of 256 dims
(the layouts the benchmark uses), other head layouts as generic sizes.
"""
from __future__ import annotations

import ctypes as C
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "suzuqu-engine-4exp_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import q4kv  # noqa: E402

F32, F16, Q8 = 0, 1, 2
WIDTH, N_SINK, N_RECENT, N_FAR = 2051, 3, 512, 1536
OUTLIERS = (3, 77, 150, 201)
RATIO, K_BLK, IDX_HD, IDX_HEADS = 4, 512, 128, 4
N_ROT, ROPE_BASE, EPS = 64, 1.0e7, 1.0e-6
DEV = "cuda"


# ------------------------------------------------------------------ cases

def listed():
    return [
        # the first tokens of a chat turn: one layer, no indexer yet
        dict(name="eager_q8", family="eager", kind=Q8, n_head=24, n_kvh=2, hd=256, ctx=1500),
        # a batch-1 engine's decode token deep in a long document
        dict(name="token_q8_128k", family="token", n_head=24, n_kvh=2, hd=256, layers=12,
             ctx=131002),
        # all 12 attention layers' steps of one sequence in one call, raw Q/K
        dict(name="step_prep_q8_layers", family="step", kind=Q8, n_head=16, n_kvh=2, hd=256,
             items=12, lo=200000, hi=200000, sparse=True, prep=True),
        # a serving batch of ragged sequences, one layer
        dict(name="step_q8_32seq", family="step", kind=Q8, n_head=16, n_kvh=2, hd=256, items=32,
             lo=8192, hi=131072, sparse=True, prep=False),
        # the f16 cache option, a small batch
        dict(name="step_f16_8seq", family="step", kind=F16, n_head=24, n_kvh=2, hd=256, items=8,
             lo=4096, hi=65536, sparse=True, prep=False),
        # a model with 128-dim heads and no selection: dense serving batch
        dict(name="step_f16_hd128_dense", family="step", kind=F16, n_head=32, n_kvh=8, hd=128,
             items=16, lo=1000, hi=16000, sparse=False, prep=False),
        # one 512-token slice of a long prompt, lists shared by the KV heads
        dict(name="prefill_q8_slice512", family="prefill", kind=Q8, n_head=24, n_kvh=2, hd=256,
             n_tok=512, base=32768, sparse=True, per_kvh=False, prep=True),
        # a whole 8192-token chunk after a 16384-token cache
        dict(name="prefill_q8_chunk8192", family="prefill", kind=Q8, n_head=16, n_kvh=2, hd=256,
             n_tok=8192, base=16384, sparse=True, per_kvh=True, prep=False),
        # a new prompt that still fits the dense window
        dict(name="prefill_q8_dense2048", family="prefill", kind=Q8, n_head=24, n_kvh=2, hd=256,
             n_tok=2048, base=0, sparse=False, per_kvh=False, prep=False),
        # the f16 cache option, a follow-up prompt of odd length, dense
        dict(name="prefill_f16_dense777", family="prefill", kind=F16, n_head=16, n_kvh=2, hd=256,
             n_tok=777, base=3333, sparse=False, per_kvh=False, prep=False),
        # the indexer of one 512-token prompt slice
        dict(name="index_prefill_512", family="index_prefill", n_tok=512, base=24576),
        # the indexer of a decode batch of ragged sequences
        dict(name="index_batch_16", family="index_batch", items=16, lo=30000, hi=262000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng):
    """(n_head, n_kvh, hd): mostly the layouts of the benchmark."""
    hd = rng.choice((256, 256, 256, 128, 64))
    if hd == 256:
        n_head, n_kvh = rng.choice(((24, 2), (24, 2), (16, 2), (16, 2), (8, 2), (16, 4)))
    elif hd == 128:
        n_head, n_kvh = rng.choice(((32, 8), (16, 2), (16, 4), (32, 4), (24, 2)))
    else:  # token rows of whole 16 bytes, as the batched calls need them
        n_head, n_kvh = rng.choice(((32, 8), (16, 4), (32, 4)))
    return n_head, n_kvh, hd


def draw(rng):
    family = rng.choice(("eager", "token", "step", "step", "step", "prefill", "prefill",
                         "prefill", "index_prefill", "index_batch"))
    n_head, n_kvh, hd = _heads(rng)
    kind = rng.choice((Q8, Q8, Q8, F16, F16, F32))
    if family == "eager":
        return dict(family=family, kind=kind, n_head=n_head, n_kvh=n_kvh, hd=hd,
                    ctx=_log(rng, 1, 2050))
    if family == "token":
        return dict(family=family, n_head=rng.choice((24, 16)), n_kvh=2, hd=256,
                    layers=rng.choice((1, 4, 12)), ctx=_log(rng, 2100, 200000))
    if family == "step":
        lo = _log(rng, 64, 20000)
        sparse = rng.random() < 0.6
        prep = sparse and kind == Q8 and hd == 256 and n_head // n_kvh <= 8 and rng.random() < 0.4
        return dict(family=family, kind=kind, n_head=n_head, n_kvh=n_kvh, hd=hd,
                    items=_log(rng, 1, 48), lo=lo, hi=_log(rng, lo, lo * (6 if sparse else 2)),
                    sparse=sparse, prep=prep)
    if family == "prefill":
        if kind == F32 and rng.random() < 0.5:
            kind = Q8
        sparse = hd == 256 and rng.random() < 0.5
        n_tok = _log(rng, 2, 2500 if kind != F32 else 600)
        base = rng.choice((0, _log(rng, 1, 8000))) if not sparse else _log(rng, 2100, 60000)
        return dict(family=family, kind=kind, n_head=n_head, n_kvh=n_kvh, hd=hd, n_tok=n_tok,
                    base=base, sparse=sparse, per_kvh=sparse and rng.random() < 0.3,
                    prep=sparse and rng.random() < 0.5)
    if family == "index_prefill":
        return dict(family=family, n_tok=_log(rng, 4, 700), base=_log(rng, 2400, 120000))
    lo = _log(rng, 2400, 200000)
    return dict(family=family, items=_log(rng, 1, 32), lo=lo, hi=_log(rng, lo, 262000))


# ----------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)


def _vectors(g, *shape):
    """N(0, 1) rows [..., hd] with the outlier channels."""
    x = _normal(g, *shape)
    for c in OUTLIERS:
        if c < shape[-1]:
            x[..., c] *= 8.0
    return x


def _q8(x):
    """q8_0 bytes [..., hd/32*34] of fp32 rows [..., hd], every rounding that
    of IEEE binary32 (formed in 64 bits and rounded once)."""
    b = x.reshape(*x.shape[:-1], -1, 32).double()
    amax = b.abs().amax(-1, keepdim=True)
    d = (amax / 127.0).float()
    inv = torch.where(d > 0, (1.0 / d.double()).float(), torch.zeros_like(d))
    q = (b * inv.double()).float().round().clamp(-127, 127).to(torch.int8)
    out = torch.cat([d.half().view(torch.uint8), q.view(torch.uint8)], -1)
    return out.reshape(*x.shape[:-1], -1)


def _store(kind, x):
    """Cache bytes of fp32 rows [..., hd]."""
    if kind == Q8:
        return _q8(x)
    return (x.half() if kind == F16 else x.contiguous()).view(torch.uint8)


def _load(kind, rows):
    """Cache bytes [..., row] -> values in 64 bits [..., hd]."""
    if kind == F16:
        return rows.contiguous().view(torch.float16).double()
    if kind == F32:
        return rows.contiguous().view(torch.float32).double()
    b = rows.reshape(*rows.shape[:-1], -1, 34)
    d = b[..., :2].contiguous().view(torch.float16).double()
    return (b[..., 2:].contiguous().view(torch.int8).double() * d).reshape(*rows.shape[:-1], -1)


def _row_bytes(kind, hd):
    return hd // 32 * 34 if kind == Q8 else hd * (2 if kind == F16 else 4)


def _fill(g, kind, n_pos, n_kvh, hd):
    """A cache [n_pos][n_kvh][row]: distinct rows up to 16384 positions, then
    those repeated (addresses, not values, are what a long cache adds)."""
    some = min(n_pos, 16384)
    rows = _store(kind, _vectors(g, some, n_kvh, hd))
    out = torch.empty(n_pos, n_kvh, rows.shape[-1], dtype=torch.uint8, device=DEV)
    for at in range(0, n_pos, some):
        out[at:at + some] = rows[:min(some, n_pos - at)]
    return out


def _far(g, rows, n, lo, hi):
    """Per row n distinct ascending values of [lo, hi[row]): one of each of n
    equal strata (hi - lo >= n)."""
    i = torch.arange(n + 1, device=DEV, dtype=torch.int64)
    edge = (i[None, :] * (hi[:, None] - lo)) // n
    u = torch.rand((rows, n), generator=g, device=DEV, dtype=torch.float64)
    wide = (edge[:, 1:] - edge[:, :-1]).double()
    return lo + edge[:, :-1] + (u * wide).long()


def _selection(g, pos):
    """Selections [len(pos)][2051] int32 of queries at positions pos: sinks +
    recent + far ones; the dense prefix where the context fits."""
    n = pos.numel()
    pos = pos.long()
    w = torch.arange(WIDTH, device=DEV)
    dense = torch.where(w[None, :] <= pos[:, None], w[None, :].expand(n, -1),
                        torch.full((1, 1), -1, device=DEV))
    long_pos = pos.clamp(min=WIDTH)
    far = _far(g, n, N_FAR, N_SINK, long_pos - N_RECENT + 1)
    recent = long_pos[:, None] - (N_RECENT - 1) + torch.arange(N_RECENT, device=DEV)[None, :]
    sinks = torch.arange(N_SINK, device=DEV)[None, :].expand(n, -1)
    sel = torch.cat([sinks, far, recent], 1)
    return torch.where((pos >= WIDTH)[:, None], sel, dense).int().contiguous()


def _block_selection(g, pos):
    """Selections as the indexer emits them: 512 ascending blocks of four
    (the first, the 128 most recent complete ones, 383 others), the causal
    tail, -1; the dense prefix where every block fits."""
    n = pos.numel()
    pos = pos.long()
    vis = (pos + 1) // RATIO
    w = torch.arange(WIDTH, device=DEV)
    dense = torch.where(w[None, :] <= pos[:, None], w[None, :].expand(n, -1),
                        torch.full((1, 1), -1, device=DEV))
    lv = vis.clamp(min=K_BLK + 1)
    n_far = K_BLK - 1 - 128
    far = _far(g, n, n_far, 1, lv - 128)
    recent = lv[:, None] - 128 + torch.arange(128, device=DEV)[None, :]
    blk = torch.cat([torch.zeros(n, 1, device=DEV, dtype=torch.int64), far, recent], 1)
    p = (blk[:, :, None] * RATIO + torch.arange(RATIO, device=DEV)).reshape(n, -1)
    tail = lv[:, None] * RATIO + torch.arange(RATIO - 1, device=DEV)[None, :]
    tail = torch.where(tail <= pos[:, None], tail, torch.full_like(tail, -1))
    sel = torch.cat([p, tail], 1)
    return torch.where((vis > K_BLK)[:, None], sel, dense).int().contiguous()


def _freq():
    """fp32 RoPE frequencies of the N_ROT/2 pairs."""
    e = -(torch.arange(N_ROT // 2, device=DEV, dtype=torch.float64) / (N_ROT // 2)).float()
    return torch.pow(torch.tensor(ROPE_BASE, device=DEV, dtype=torch.float64), e.double()).float()


def _prep(x, w, pos):
    """RMSNorm * w, then RoPE of the first N_ROT dims' adjacent pairs at pos
    (one position per leading index), in 64 bits; the angle is the fp32
    product that defines it."""
    x = x.double()
    x = x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()
    ang = (pos.double()[:, None] * _freq().double()[None, :]).float().double()
    while ang.dim() < x.dim():
        ang = ang.unsqueeze(1)
    c, s = torch.cos(ang), torch.sin(ang)
    a, b = x[..., 0:N_ROT:2].clone(), x[..., 1:N_ROT:2].clone()
    x = x.clone()
    x[..., 0:N_ROT:2] = a * c - b * s
    x[..., 1:N_ROT:2] = a * s + b * c
    return x


def _pool(raw):
    """Pooled block keys (64 bits) of raw fp16 keys [n*RATIO][128], w = 1."""
    m = raw.double().reshape(-1, RATIO, IDX_HD).mean(1)
    pos = torch.arange(m.shape[0], device=DEV) * RATIO
    return _prep(m, torch.ones(IDX_HD, device=DEV), pos)


# ---------------------------------------------------------------- prepare

class State:
    """Buffers of one case and the calls of one pass: (function, arguments)."""

    def __init__(self):
        self.calls, self.out, self.keep = [], None, []


_rt = None


def _lib():
    global _rt
    if _rt is None:
        _rt = q4kv.Runtime()
    return _rt.lib


def _p(t, off=0):
    return C.c_void_p(t.data_ptr() + off)


def _call(st, name, *args):
    st.calls.append((getattr(_lib(), name), args))


def prepare(case, seed):
    _lib()
    st = State()
    globals()["_prepare_" + case["family"]](st, case, _inputs(case, seed))
    torch.cuda.synchronize()
    return st


def run(state):
    for fn, args in state.calls:
        if fn(*args) is False:
            raise RuntimeError(f"{fn.__name__} failed")
    return state.out


def _inputs(case, seed):
    return globals()["_inputs_" + case["family"]](case, _gen(seed))


def _u32(v):
    return C.c_uint32(int(v))


def _f(v):
    return C.c_float(v)


def _scale(case):
    return 1.0 / math.sqrt(case["hd"])


# eager: cache rows 0..ctx-1 hold the context, the new token goes to ctx

def _inputs_eager(case, g):
    nk, hd = case["n_kvh"], case["hd"]
    return dict(kc=_fill(g, case["kind"], case["ctx"] + 1, nk, hd),
                vc=_fill(g, case["kind"], case["ctx"] + 1, nk, hd),
                k=_vectors(g, nk, hd), v=_vectors(g, nk, hd),
                q=_vectors(g, case["n_head"], hd), gate=_normal(g, case["n_head"], hd))


def _prepare_eager(st, case, x):
    kind, nk, hd, ctx = case["kind"], case["n_kvh"], case["hd"], case["ctx"]
    out = torch.empty(case["n_head"], hd, device=DEV)
    at = ctx * nk * _row_bytes(kind, hd)
    write = {Q8: "q4_hip_f32_to_q8", F16: "q4_hip_f32_to_f16", F32: "q4_hip_copy"}[kind]
    for c, new in ((x["kc"], x["k"]), (x["vc"], x["v"])):
        _call(st, write, _p(c, at), _p(new), C.c_uint64(nk * hd))
    _call(st, "q4_hip_qsa_decode", _p(x["q"]), _p(x["kc"]), _p(x["vc"]), _p(x["gate"]), _p(out),
          _u32(case["n_head"]), _u32(nk), _u32(hd), _u32(ctx + 1), _u32(ctx + 1),
          _f(_scale(case)), C.c_int(kind))
    st.keep = x
    st.out = [out, x["kc"][ctx], x["vc"][ctx]]


# token: 12 layers one after the other, positions 0..ctx-1 held, token at ctx

def _inputs_token(case, g):
    nk, hd, ctx, n_layer = case["n_kvh"], case["hd"], case["ctx"], case["layers"]
    nb = (ctx + 1 + RATIO - 1) // RATIO + 1
    layers = []
    for _ in range(n_layer):
        raw = _normal(g, nb * RATIO, IDX_HD).half()
        layers.append(dict(
            kc=_fill(g, Q8, ctx + 1, nk, hd), vc=_fill(g, Q8, ctx + 1, nk, hd),
            k=_vectors(g, nk, hd), v=_vectors(g, nk, hd), q=_vectors(g, case["n_head"], hd),
            gate=_normal(g, case["n_head"], hd), raw=raw, pool=_pool(raw).float(),
            ik=_normal(g, IDX_HD), iq=_normal(g, IDX_HEADS, IDX_HD),
            wk=torch.ones(IDX_HD, device=DEV), wq=torch.ones(IDX_HD, device=DEV)))
    return dict(layers=layers, nb=nb)


def _prepare_token(st, case, x):
    nk, hd, ctx, nh = case["n_kvh"], case["hd"], case["ctx"], case["n_head"]
    n_layer, nb, vis = case["layers"], x["nb"], (case["ctx"] + 1) // RATIO
    out = torch.empty(n_layer, nh, hd, device=DEV)
    score = torch.zeros(n_layer, nb, device=DEV)
    sel = torch.zeros(n_layer, WIDTH, device=DEV, dtype=torch.int32)
    _call(st, "q4_hip_pos_push", C.c_int32(ctx))
    for i, y in enumerate(x["layers"]):
        _call(st, "q4_hip_kv_append_d", _p(y["kc"]), _p(y["vc"]), _p(y["k"]), _p(y["v"]),
              _u32(nk * hd), _u32(nk * _row_bytes(Q8, hd)), C.c_int(Q8))
        _call(st, "q4_hip_qsa_index_score_d", _p(y["raw"]), _p(y["pool"]), _p(y["wk"]),
              _p(y["ik"]), _p(y["iq"]), _p(y["wq"]), _p(score[i]), _u32(nb), _u32(IDX_HEADS),
              _u32(IDX_HD), _u32(RATIO), _u32(N_ROT), _f(ROPE_BASE), _f(EPS))
        _call(st, "q4_hip_qsa_topk_d", _p(score[i]), _p(sel[i]), _u32(nb), _u32(K_BLK),
              _u32(RATIO), _u32(WIDTH))
        _call(st, "q4_hip_qsa_decode_idx", _p(y["q"]), _p(y["kc"]), _p(y["vc"]), _p(y["gate"]),
              _p(out[i]), _p(sel[i]), _u32(WIDTH), _u32(nh), _u32(nk), _u32(hd), _u32(1),
              _u32(ctx + 1), _f(_scale(case)), C.c_int(Q8))
    st.keep = x
    st.out = [out, score[:, :vis], sel, [y["raw"][ctx] for y in x["layers"]],
              [y["kc"][ctx] for y in x["layers"]], [y["vc"][ctx] for y in x["layers"]]]


# step: each item's cache ends at its new token's row, which is the last row
# of its slot of hi + 1 positions

def _inputs_step(case, g):
    nk, hd, nh, n = case["n_kvh"], case["hd"], case["n_head"], case["items"]
    lo, hi, kind = case["lo"], case["hi"], case["kind"]
    t = torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    pos = (lo * (hi / lo) ** t).round().long().clamp(lo, hi)  # log-uniform lengths
    x = dict(pos=pos, kc=torch.empty(n, hi + 1, nk, _row_bytes(kind, hd), dtype=torch.uint8,
                                     device=DEV))
    x["vc"] = torch.empty_like(x["kc"])
    for i in range(n):
        x["kc"][i] = _fill(g, kind, hi + 1, nk, hd)
        x["vc"][i] = _fill(g, kind, hi + 1, nk, hd)
    x.update(k=_vectors(g, n, nk, hd), v=_vectors(g, n, nk, hd), q=_vectors(g, n, nh, hd),
             gate=_normal(g, n, nh, hd))
    if case["sparse"]:
        x["sel"] = _selection(g, pos.repeat_interleave(nk)).reshape(n, nk, WIDTH)
    if case["prep"]:
        x["wq"] = 1.0 + 0.1 * _normal(g, n, hd)
        x["wk"] = 1.0 + 0.1 * _normal(g, n, hd)
    return x


def _prepare_step(st, case, x):
    nk, hd, nh, n = case["n_kvh"], case["hd"], case["n_head"], case["items"]
    kind, hi = case["kind"], case["hi"]
    bpt = nk * _row_bytes(kind, hd)
    pos = x["pos"].tolist()
    out = torch.empty(n, nh, hd, device=DEV)
    prep = case["prep"]
    if prep:
        x["qg"] = torch.cat([x["q"], x["gate"]], -1).contiguous()
        x["g_out"] = torch.empty(n, nh, hd, device=DEV)
    descs = ((q4kv.PrepStepDesc if prep else q4kv.StepDesc) * n)()
    for i in range(n):
        s = descs[i].step if prep else descs[i]
        at = (i * (hi + 1) + hi - pos[i]) * bpt
        s.seq.kcache, s.seq.vcache = x["kc"].data_ptr() + at, x["vc"].data_ptr() + at
        s.seq.q = (x["qg"] if prep else x["q"])[i].data_ptr()
        s.seq.gate = (x["g_out"] if prep else x["gate"])[i].data_ptr()
        s.seq.out = out[i].data_ptr()
        s.seq.idx = x["sel"][i].data_ptr() if case["sparse"] else None
        s.seq.n_sel = WIDTH if case["sparse"] else pos[i] + 1
        s.seq.idx_kvh_stride, s.seq.max_kv = WIDTH, pos[i] + 1
        s.k, s.v, s.pos = x["k"][i].data_ptr(), x["v"][i].data_ptr(), pos[i]
        if prep:
            descs[i].wn_q, descs[i].wn_k = x["wq"][i].data_ptr(), x["wk"][i].data_ptr()
    d = torch.from_numpy(np.frombuffer(bytes(descs), dtype=np.uint8).copy()).to(DEV)
    max_n = WIDTH if case["sparse"] else max(pos) + 1
    args = [_p(d), _u32(n), _u32(nh), _u32(nk), _u32(hd), _f(_scale(case)), C.c_int(kind),
            _u32(max_n)]
    if prep:
        _call(st, "q4_hip_qsa_step_prep_batch", *args, _u32(N_ROT), _f(ROPE_BASE), _f(EPS))
    else:
        _call(st, "q4_hip_qsa_step_batch", *args)
    st.keep = (x, d)
    st.out = [out, x["kc"][:, hi], x["vc"][:, hi]]


# prefill: positions 0..base-1 held, the slice's tokens at base..

def _inputs_prefill(case, g):
    nk, hd, nh, n = case["n_kvh"], case["hd"], case["n_head"], case["n_tok"]
    base, kind = case["base"], case["kind"]
    x = dict(kc=_fill(g, kind, base + n, nk, hd), vc=_fill(g, kind, base + n, nk, hd),
             k=_vectors(g, n, nk, hd), v=_vectors(g, n, nk, hd), q=_vectors(g, n, nh, hd),
             gate=_normal(g, n, nh, hd))
    if case["sparse"]:
        pos = base + torch.arange(n, device=DEV)
        if case["per_kvh"]:
            x["sel"] = _selection(g, pos.repeat_interleave(nk)).reshape(n, nk, WIDTH)
        else:
            x["sel"] = _block_selection(g, pos)
    if case["prep"]:
        x["wq"] = 1.0 + 0.1 * _normal(g, hd)
    return x


def _prepare_prefill(st, case, x):
    nk, hd, nh, n = case["n_kvh"], case["hd"], case["n_head"], case["n_tok"]
    base, kind = case["base"], case["kind"]
    out = torch.empty(n, nh, hd, device=DEV)
    q, gate = x["q"], x["gate"]
    st.out = [out, x["kc"][base:], x["vc"][base:]]
    if case["prep"]:
        qg = torch.cat([q, gate], -1).contiguous()
        x["qg"], x["q"], x["gate"] = qg, torch.empty_like(q), torch.empty_like(gate)
        q, gate = x["q"], x["gate"]
        _call(st, "q4_hip_qsa_q_prep_n", _p(qg), _p(x["wq"]), _p(q), _p(gate), _u32(nh),
              _u32(hd), _u32(N_ROT), C.c_int32(base), _f(ROPE_BASE), _f(EPS), _u32(n))
        st.out += [q, gate]
    cache = q4kv.KvCache(kind=kind, n_layer=1, n_kvh=nk, hd=hd, max_kv=base + n,
                         bpt=nk * _row_bytes(kind, hd), n_kv=base,
                         d_k=x["kc"].data_ptr(), d_v=x["vc"].data_ptr())
    c = C.byref(cache)
    _call(st, "q4kv_write_chunk", c, _u32(0), _u32(base), _p(x["k"]), _p(x["v"]), _u32(n))
    sel = _p(x["sel"]) if case["sparse"] else C.c_void_p(None)
    _call(st, "q4kv_attend", c, _u32(0), _p(q), _p(gate), _p(out), _u32(nh), _u32(n),
          _u32(base), sel, _u32(WIDTH), C.c_uint64(WIDTH * (nk if case["per_kvh"] else 1)),
          C.c_uint64(WIDTH if case["per_kvh"] else 0))
    st.keep = (x, cache)


# index_prefill: base positions pooled already, the slice's raw keys arrive

def _inputs_index_prefill(case, g):
    n, base = case["n_tok"], case["base"]
    nb = (base + n) // RATIO
    raw = _normal(g, base + n + RATIO, IDX_HD).half()
    return dict(raw=raw, pool=_pool(raw[:nb * RATIO]).float().contiguous(),
                new=_normal(g, n, IDX_HD), q=_normal(g, n, IDX_HEADS, IDX_HD),
                wn=torch.ones(IDX_HD, device=DEV))


def _prepare_index_prefill(st, case, x):
    n, base = case["n_tok"], case["base"]
    b0, nb = base // RATIO, (base + n) // RATIO
    score = torch.zeros(n, nb, device=DEV)
    sel = torch.zeros(n, WIDTH, device=DEV, dtype=torch.int32)
    _call(st, "q4_hip_f32_to_f16", _p(x["raw"], base * IDX_HD * 2), _p(x["new"]),
          C.c_uint64(n * IDX_HD))
    if nb > b0:
        _call(st, "q4_hip_qsa_pool", _p(x["raw"]), _p(x["pool"]), _p(x["wn"]), _u32(IDX_HD),
              _u32(RATIO), _u32(b0), _u32(nb), _u32(N_ROT), _f(ROPE_BASE), _f(EPS))
    _call(st, "q4_hip_qsa_score", _p(x["q"]), _p(x["pool"]), _p(score), _u32(n), _u32(nb),
          _u32(nb), _u32(IDX_HEADS), _u32(IDX_HD), _u32(base), _u32(RATIO))
    _call(st, "q4_hip_qsa_topk", _p(score), _p(sel), _u32(n), _u32(nb), _u32(nb), _u32(K_BLK),
          _u32(RATIO), _u32(base), _u32(WIDTH))
    st.keep = x
    # blocks that every token sees, and the causal rest (masked by -1e30)
    st.out = [score[:, :b0], score[:, b0:], sel, x["pool"][b0:], x["raw"][base:base + n]]


# index_batch: item i holds positions 0..pos[i]-1, its new token at pos[i]

def _inputs_index_batch(case, g):
    n, lo, hi = case["items"], case["lo"], case["hi"]
    t = torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    pos = (lo * (hi / lo) ** t).round().long().clamp(lo, hi)
    nb = (hi + 1 + RATIO - 1) // RATIO + 1
    raw = torch.empty(n, nb * RATIO, IDX_HD, device=DEV, dtype=torch.float16)
    pool = torch.empty(n, nb, IDX_HD, device=DEV)
    for i in range(n):
        raw[i] = _normal(g, nb * RATIO, IDX_HD).half()
        pool[i] = _pool(raw[i]).float()
    return dict(pos=pos, nb=nb, raw=raw, pool=pool, k=_normal(g, n, IDX_HD),
                q=_normal(g, n, IDX_HEADS, IDX_HD), w=torch.ones(IDX_HD, device=DEV))


def _prepare_index_batch(st, case, x):
    n, nb = case["items"], x["nb"]
    pos = x["pos"].tolist()
    score = torch.zeros(n, nb, device=DEV)
    sel = torch.zeros(n, WIDTH, device=DEV, dtype=torch.int32)
    descs = (q4kv.IndexDesc * n)()
    w = x["w"].data_ptr()
    for i in range(n):
        d = descs[i]
        d.raw, d.pool = x["raw"][i].data_ptr(), x["pool"][i].data_ptr()
        d.wn_k, d.wn_q, d.k_new, d.q = w, w, x["k"][i].data_ptr(), x["q"][i].data_ptr()
        d.score, d.sel, d.pos = score[i].data_ptr(), sel[i].data_ptr(), pos[i]
    dev = torch.from_numpy(np.frombuffer(bytes(descs), dtype=np.uint8).copy()).to(DEV)
    _call(st, "q4_hip_qsa_index_batch", _p(dev), _u32(n), _u32((max(pos) + 1) // RATIO),
          _u32(IDX_HEADS), _u32(IDX_HD), _u32(RATIO), _u32(N_ROT), _f(ROPE_BASE), _f(EPS),
          _u32(K_BLK), _u32(WIDTH))
    st.keep = (x, dev)
    st.out = [score, sel] + ([x["raw"][i, pos[i]] for i in range(n)] if n <= 32 else [])


# ------------------------------------------------------------------- work

def _lengths(case):
    """Attended positions per token of the prefill families, summed."""
    n, base = case["n_tok"], case["base"]
    if not case["sparse"]:
        return n * base + n * (n + 1) // 2
    return sum(min(WIDTH, base + t + 1) for t in range(n))


def work(case):
    f = case["family"]
    if f in ("index_prefill", "index_batch"):
        if f == "index_prefill":
            n, nb = case["n_tok"], (case["base"] + case["n_tok"]) // RATIO
            new = nb - case["base"] // RATIO
            byte = (n * IDX_HD * 6 + new * IDX_HD * (2 * RATIO + 4) + nb * IDX_HD * 4
                    + n * IDX_HEADS * IDX_HD * 4 + n * nb * 4 + n * WIDTH * 4)
            return dict(bytes=byte, flops=2 * n * nb * IDX_HEADS * IDX_HD)
        n, lo, hi = case["items"], case["lo"], case["hi"]
        mean = (hi - lo) / math.log(hi / lo) if hi > lo else lo
        nb = n * mean / RATIO
        return dict(bytes=nb * (IDX_HD + 1) * 4 + n * (WIDTH * 4 + IDX_HEADS * IDX_HD * 4),
                    flops=2 * nb * IDX_HEADS * IDX_HD)
    nk, hd, nh, kind = case["n_kvh"], case["hd"], case["n_head"], case.get("kind", Q8)
    row = nk * _row_bytes(kind, hd)
    qo = 3 * nh * hd * 4  # query and gate in, output out
    new = 2 * (nk * hd * 4 + row)  # the token's K and V rows in and stored
    if f == "eager":
        n = case["ctx"] + 1
        return dict(bytes=2 * n * row + qo + new, flops=4 * nh * hd * n)
    if f == "token":
        n, n_layer = min(WIDTH, case["ctx"] + 1), case["layers"]
        nb = (case["ctx"] + 1) // RATIO
        byte = 2 * n * row + qo + new + nb * (IDX_HD + 1) * 4 + WIDTH * 8
        return dict(bytes=n_layer * byte,
                    flops=n_layer * (4 * nh * hd * n + 2 * nb * IDX_HEADS * IDX_HD))
    if f == "step":
        lo, hi = case["lo"], case["hi"]
        n = (hi - lo) / math.log(hi / lo) if hi > lo else lo
        if case["sparse"]:
            n = min(WIDTH, n)
        idx = nk * WIDTH * 4 if case["sparse"] else 0
        prep = nh * hd * 4 if case["prep"] else 0
        return dict(bytes=case["items"] * (2 * n * row + qo + new + idx + prep),
                    flops=case["items"] * 4 * nh * hd * n)
    n, pairs = case["n_tok"], _lengths(case)
    idx = n * WIDTH * 4 * (nk if case["per_kvh"] else 1) if case["sparse"] else 0
    prep = 2 * n * nh * hd * 4 if case["prep"] else 0
    return dict(bytes=2 * (case["base"] + n) * row + n * (qo + new) + idx + prep,
                flops=4 * nh * hd * pairs)


def tolerance(case):
    """Attention and scores in 32 bits: the results are up to 1.1e-5
    (attention) and 2.5e-5 (scores of a prompt slice) off 64 bits, four times
    that is allowed. Where selections are computed too, a rounding of two
    close scores swaps blocks, and with them rows of the attention."""
    f = case["family"]
    if f == "token":
        return {"rel": 3e-2, "max": 0.9, "differ": 1e-2}
    if f in ("index_prefill", "index_batch"):
        return {"rel": 1e-4, "max": 4e-3, "differ": 1e-2}
    return {"rel": 5e-5, "max": 4e-3, "differ": 1e-5}


# ------------------------------------------------------------------ exact

def _attend64(q, k, v, scale, gate, mask):
    """q [n][g][hd], k and v [n or 1][len][hd], mask [n][len] (True = seen)."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    s = s.masked_fill(~mask[:, None, :], -math.inf)
    o = torch.matmul(torch.softmax(s, -1), v)
    return o * torch.sigmoid(gate)


def exact(case, seed):
    x = _inputs(case, seed)
    f = case["family"]
    if f == "index_prefill":
        n, base = case["n_tok"], case["base"]
        b0, nb = base // RATIO, (base + n) // RATIO
        x["raw"][base:base + n] = x["new"].half()
        x["pool"][b0:] = _pool(x["raw"][:nb * RATIO])[b0:].float()
        p, q = x["pool"].double(), x["q"].double()
        score = torch.zeros(n, nb, device=DEV, dtype=torch.float64)
        for h in range(IDX_HEADS):
            score += torch.matmul(q[:, h], p.t().contiguous()).clamp(min=0)
        vis = (base + torch.arange(n, device=DEV) + 1) // RATIO
        score[torch.arange(nb, device=DEV)[None, :] >= vis[:, None]] = -1.0e30
        return [score[:, :b0], score[:, b0:], None, p[b0:],
                x["raw"][base:base + n].double()]
    if f == "index_batch":
        n, nb, pos = case["items"], x["nb"], x["pos"].tolist()
        score = torch.zeros(n, nb, device=DEV, dtype=torch.float64)
        for i in range(n):
            score[i, :(pos[i] + 1) // RATIO] = _decode_scores(
                x["raw"][i], x["pool"][i], x["k"][i], x["q"][i], x["w"], pos[i])
        return [score, None] + ([x["raw"][i, pos[i]].double() for i in range(n)]
                                if n <= 32 else [])
    nk, hd, nh, kind = case["n_kvh"], case["hd"], case["n_head"], case.get("kind", Q8)
    gqa, scale = nh // nk, _scale(case)
    if f == "token":
        score = torch.stack([_decode_scores(y["raw"], y["pool"], y["ik"], y["iq"], y["wq"],
                                            case["ctx"]) for y in x["layers"]])
        # the selection, and with it the attention, is the program's own
        return [None, score, None, [y["raw"][case["ctx"]].double() for y in x["layers"]],
                None, None]
    if f == "eager":
        x["kc"][-1], x["vc"][-1] = _store(kind, x["k"]), _store(kind, x["v"])
        k, v = _load(kind, x["kc"]).transpose(0, 1), _load(kind, x["vc"]).transpose(0, 1)
        mask = torch.ones(nk, k.shape[1], device=DEV, dtype=torch.bool)
        out = _attend64(x["q"].double().reshape(nk, gqa, hd), k, v.contiguous(), scale,
                        x["gate"].double().reshape(nk, gqa, hd), mask)
        return [out.reshape(nh, hd), None, None]
    if f == "step":
        hi, pos, outs = case["hi"], x["pos"].tolist(), []
        for i in range(case["items"]):
            q, k = x["q"][i].double(), x["k"][i]
            if case["prep"]:
                at = torch.tensor([pos[i]], device=DEV)
                q = _prep(q[None], x["wq"][i], at)[0].float().double()
                k = _prep(k[None], x["wk"][i], at)[0].float()
            kc, vc = x["kc"][i, hi - pos[i]:], x["vc"][i, hi - pos[i]:]
            kc[pos[i]], vc[pos[i]] = _store(kind, k), _store(kind, x["v"][i])
            if case["sparse"]:
                sel = x["sel"][i].long()
                mask, sel, h = sel >= 0, sel.clamp(min=0), torch.arange(nk, device=DEV)[:, None]
                kk, vv = _load(kind, kc[sel, h]), _load(kind, vc[sel, h])
            else:
                kk, vv = (_load(kind, c).transpose(0, 1).contiguous() for c in (kc, vc))
                mask = torch.ones(nk, kk.shape[1], device=DEV, dtype=torch.bool)
            outs.append(_attend64(q.reshape(nk, gqa, hd), kk, vv, scale,
                                  x["gate"][i].double().reshape(nk, gqa, hd), mask))
        return [torch.stack(outs).reshape(-1, nh, hd), None, None]
    n, base = case["n_tok"], case["base"]
    x["kc"][base:], x["vc"][base:] = _store(kind, x["k"]), _store(kind, x["v"])
    kk, vv = _load(kind, x["kc"]), _load(kind, x["vc"])
    q, gate = x["q"].double(), x["gate"].double()
    if case["prep"]:
        q = _prep(q, x["wq"], base + torch.arange(n, device=DEV))
    q32 = q.float().double()
    out = torch.empty(n, nh, hd, device=DEV, dtype=torch.float64)
    step = 32 if case["sparse"] else 256
    for h in range(nk):
        hs = slice(h * gqa, (h + 1) * gqa)
        kh, vh = kk[:, h].contiguous(), vv[:, h].contiguous()
        for t in range(0, n, step):
            u = min(n, t + step)
            if case["sparse"]:
                sel = (x["sel"][t:u, h] if case["per_kvh"] else x["sel"][t:u]).long()
                mask, at = sel >= 0, sel.clamp(min=0)
                out[t:u, hs] = _attend64(q32[t:u, hs], kh[at], vh[at], scale, gate[t:u, hs], mask)
            else:
                end = base + u
                see = torch.arange(end, device=DEV)[None, :] <= base + torch.arange(
                    t, u, device=DEV)[:, None]
                qq = q32[t:u, hs].transpose(0, 1).contiguous()
                s = torch.matmul(qq, kh[:end].t().contiguous()) * scale
                s = torch.softmax(s.masked_fill(~see[None], -math.inf), -1)
                out[t:u, hs] = torch.matmul(s, vh[:end]).transpose(0, 1) * torch.sigmoid(
                    gate[t:u, hs])
    return [out, None, None] + ([q, gate] if case["prep"] else [])


def _decode_scores(raw, pool, k, q, w, pos):
    """Scores (64 bits) of the blocks visible at pos after the new key."""
    raw[pos] = k.half()
    vis = (pos + 1) // RATIO
    if (pos + 1) % RATIO == 0:
        pool[vis - 1] = _pool(raw[:vis * RATIO])[vis - 1].float()
    q = _prep(q[None], w, torch.tensor([pos], device=DEV))[0].float().double()
    return torch.matmul(pool[:vis].double(), q.t().contiguous()).clamp(min=0).sum(-1)
