"""Block scores of a prompt chunk (>= 4 tokens): the matrix-pipe kernel against
float64 over the edges of its three tile sizes, every head count, output
rows that are not 16-byte aligned, and rows of very different magnitudes.

Both operands are split into two fp16 parts, rounded to nearest after each row
is multiplied by a power of two that brings its largest magnitude to 2^14 or
more: hi is within 2^-11 of its element, lo rounds what is left to 2^-22 of the
element or to half fp16's smallest step, 2^-39 of the row's largest magnitude.
A product loses both roundings and lo*lo, 3 * 2^-22 of itself and 2^-39 of each
element times the other row's largest; fp32 accumulation of 384 products adds
at most 384 * 2^-24."""
import numpy as np
import pytest

from qsa_util import IDX_DIM, RATIO

pytestmark = pytest.mark.gpu


def _bound(q, pool):
    aq, ap = np.abs(q).astype(np.float64), np.abs(pool).astype(np.float64)
    return sum((3 * 2.0 ** -22 + 384 * 2.0 ** -24) * (aq[:, h] @ ap.T)
               + 2.0 ** -38 * (aq[:, h].sum(1)[:, None] * ap.max(1)
                               + aq[:, h].max(1)[:, None] * ap.sum(1))
               for h in range(q.shape[1]))


@pytest.mark.parametrize("n_tok,n_blocks,n_head,pad,offset,mag", [
    # 8 tokens x 64 blocks per workgroup: up to 256 of them
    (4, 1, 4, 0, 0, (0, 0)),
    (5, 3, 1, 1, 0, (0, 0)),           # odd row stride: single stores
    (7, 63, 3, 1, 1, (0, 0)),
    (8, 64, 4, 0, 0, (0, 0)),          # a full tile
    (9, 65, 2, 3, 0, (0, 0)),          # 68 floats per row: 16-byte stores
    (9, 65, 4, 3, 1, (0, 0)),          # the same rows off the 16-byte grid
    (70, 1031, 4, 1, 0, (30, -30)),    # queries near 1e9, pool rows near 1e-9
    (70, 1031, 4, 1, 0, (-100, 90)),
    (40, 300, 4, 0, 0, (120, -118)),
    # 16 x 128: up to 512
    (144, 1152, 4, 0, 0, (0, 0)),
    (129, 1025, 3, 1, 0, (0, 0)),
    (17, 5503, 4, 1, 0, (0, 0)),
    # 32 x 256
    (288, 4096, 4, 0, 0, (0, 0)),
    (289, 4097, 2, 3, 0, (0, 0)),
    (511, 3839, 4, 2, 1, (0, 0)),
])
def test_prefill_score(rt, n_tok, n_blocks, n_head, pad, offset, mag):
    lib = rt.lib
    rng = np.random.default_rng(n_tok * 1000 + n_blocks)
    # every row has its own magnitude, 2^-3 .. 2^3 around the case's
    sq = 2.0 ** (mag[0] + rng.integers(-3, 4, (n_tok, n_head, 1)))
    sp = 2.0 ** (mag[1] + rng.integers(-3, 4, (n_blocks, 1)))
    q = (rng.standard_normal((n_tok, n_head, IDX_DIM)) * sq).astype(np.float32)
    pool = (rng.standard_normal((n_blocks, IDX_DIM)) * sp).astype(np.float32)
    pool[n_blocks // 2] = 0.0
    q[1, 0] = 0.0
    stride = n_blocks + pad
    pos0 = max(0, (n_blocks - 1) * RATIO - n_tok // 2)  # the chunk's end sees the last block
    fill = np.float32(7.5)
    d_q, d_pool = rt.upload(q), rt.upload(pool)
    d_sc = rt.upload(np.full(n_tok * stride + offset + 4, fill, np.float32))
    assert lib.q4_hip_qsa_score(d_q, d_pool, d_sc + 4 * offset, n_tok, n_blocks, stride, n_head,
                                IDX_DIM, pos0, RATIO)
    rt.sync()
    flat = rt.download(d_sc, 4 * (n_tok * stride + offset + 4), np.float32)
    for p in (d_q, d_pool, d_sc):
        rt.free(p)
    got = flat[offset:offset + n_tok * stride].reshape(n_tok, stride)
    assert (flat[:offset] == fill).all() and (flat[offset + n_tok * stride:] == fill).all()
    assert (got[:, n_blocks:] == fill).all()

    want = sum(np.maximum(q[:, h].astype(np.float64) @ pool.T.astype(np.float64), 0)
               for h in range(n_head))
    bound = _bound(q, pool)
    n_vis = (pos0 + 1 + np.arange(n_tok)) // RATIO
    seen = np.arange(n_blocks)[None, :] < n_vis[:, None]
    assert (got[:, :n_blocks][~seen] == np.float32(-1e30)).all()
    err = np.abs(got[:, :n_blocks] - want)
    assert (err[seen] <= bound[seen]).all(), (err - bound)[seen].max()


@pytest.mark.parametrize("n_tok,n_blocks", [(9, 65), (129, 1025), (289, 4097)])
@pytest.mark.parametrize("apart", [8, 14, 18])
def test_prefill_score_large_in_different_dims(rt, n_tok, n_blocks, apart):
    """Queries whose second half and pool rows whose first half are 2^-apart of
    the other half: every product is of the small elements."""
    rng = np.random.default_rng(apart * 10000 + n_blocks)
    q = rng.standard_normal((n_tok, 4, IDX_DIM)).astype(np.float32)
    pool = rng.standard_normal((n_blocks, IDX_DIM)).astype(np.float32)
    q[..., IDX_DIM // 2:] *= np.float32(2.0 ** -apart)
    pool[:, :IDX_DIM // 2] *= np.float32(2.0 ** -apart)
    d_q, d_pool = rt.upload(q), rt.upload(pool)
    d_sc = rt.alloc(4 * n_tok * n_blocks)
    assert rt.lib.q4_hip_qsa_score(d_q, d_pool, d_sc, n_tok, n_blocks, n_blocks, 4, IDX_DIM,
                                   n_blocks * RATIO, RATIO)
    rt.sync()
    got = rt.download(d_sc, 4 * n_tok * n_blocks, np.float32).reshape(n_tok, n_blocks)
    for p in (d_q, d_pool, d_sc):
        rt.free(p)
    want = sum(np.maximum(q[:, h].astype(np.float64) @ pool.T.astype(np.float64), 0)
               for h in range(4))
    err, bound = np.abs(got - want), _bound(q, pool)
    assert (err <= bound).all(), (err - bound).max()
