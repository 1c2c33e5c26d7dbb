/*
 * q4kv_rows.hip -- decode attention at 64 and 128 head dims (q8_0 and f16
 * caches, up to 16 query heads per KV head): one token, a position list or
 * the dense prefix, per (token or sequence, KV head) item.
 *
 * Rows of 68 to 256 bytes are short enough for a wave to hold 16 positions'
 * K and V rows in registers, in the layouts the matrix products take, twice
 * over: the rows of the next pass are in flight while this pass computes,
 * and waves never wait for one another inside the loop.
 *  - scores: lane (c, g) holds K[position c][32 b + 8 g .. + 7], the A
 *    operand of S^T = K Q^T (v_mfma_f32_16x16x32_f16; columns 0-7 the fp16
 *    part of eight heads' q, 8-15 the residual); q8_0: exact int8 values in
 *    fp16, the block scales applied in fp32 to each block's product;
 *  - online softmax in base 2 per wave;
 *  - O^T += V^T P^T (16x16x16): the weights leave the score tile in the B
 *    layout (split hi / lo in the columns); lane (c, g) loads U = hd / 16
 *    consecutive dims U c .. of positions 4 g + i, and regroups them into
 *    the A operands of U tiles (tile u, row r: dim U r + u); q8_0: v x scale
 *    in two fp16 parts, exact (VScale, one for the wave).
 * An item's entries are cut into pieces of whole passes of four waves; the
 * pieces an item needs follow its own length, so a ragged batch gives every
 * workgroup the same amount of work. Items of one piece finish in place, the
 * others leave partials that a second launch merges.
 *
 * What bounds it: the cache rows from HBM. 16 sequences, 8 KV heads of 128
 * dims in f16, 1000 to 16000 positions (355 MB): 73-95 us by the lengths
 * drawn, 3.7 TB/s with the append and merge launches; the generic kernel,
 * whose workgroups walk one 64-position chunk after the other between
 * barriers, 540-680 us. Without the second set of registers (or with a
 * branch around a load, past which the compiler waits for all of them) the
 * q8_0 form took 119 us instead of 79.
 */
#include <stdlib.h>
#include <algorithm>

#include "q4kv_attn_item.h"

namespace {

typedef uint32_t u3_t __attribute__((ext_vector_type(3)));
typedef uint32_t u3u_t __attribute__((ext_vector_type(3), aligned(4)));
typedef uint32_t u2u_t __attribute__((ext_vector_type(2), aligned(4)));
typedef float fv2 __attribute__((ext_vector_type(2)));

constexpr uint32_t PASS = 16, PHEAD = 4; /* a partial row: m, l, 2 unused, hd accumulators */

struct RowArgs {
    AttnArgs a;
    uint32_t piece, S; /* entries per piece (a multiple of 64), pieces in the grid */
};

/* pieces item `it` is cut into: the last of the grid's takes what is left */
__device__ inline uint32_t pieces_of(const Item &it, const RowArgs &r) {
    const uint32_t p = (it.n + r.piece - 1u) / r.piece;
    return p < 1u ? 1u : p < r.S ? p : r.S;
}

/* (x, y) as fp16, rounded to nearest (sel 0), or what that left (sel -1), so
 * that both together hold 22 bits: weights cut off instead (split_pk) lower
 * every output by 8e-8 on average */
__device__ inline uint32_t part_pk(float x, float y, float sel) {
    const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector((fv2){x, y}, h2_t));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((fv2){fmaf(sel, h2lo(h), x), fmaf(sel, h2hi(h), y)}, h2_t));
}

/* 1024 + (byte ^ 0x80) of four bytes, in two packed fp16 pairs */
__device__ inline void biased_h4(uint32_t w, h2_t &x, h2_t &y) {
    w ^= 0x80808080u;
    x = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u));
    y = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u));
}

template <int KIND, int HD, int MODE, int HG>
__global__ __launch_bounds__(256, HG == 1 ? 3 : 2) void qsa_rows_k(RowArgs ra) {
    constexpr uint32_t NB = HD / 32, U = HD / 16, NV = KIND == Q4KV_Q8 ? 2 : 1;
    constexpr uint32_t ROWB = KIND == Q4KV_Q8 ? NB * 34 : HD * 2;
    constexpr uint32_t MROW = HD + 4; /* merge rows: [wave][head][dim] */
    const AttnArgs &a = ra.a;
    __shared__ __attribute__((aligned(16))) float mrg[4 * 8 * HG * MROW];
    __shared__ __attribute__((aligned(16))) float s_ks[4][KIND == Q4KV_Q8 ? NB * 16 : 4];
    __shared__ float s_m[4][8 * HG], s_l[4][8 * HG];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t c = lane & 15u, jg = lane >> 4;
    const uint32_t item = a.item0 + blockIdx.y, s = blockIdx.x;
    const uint32_t gqa = a.n_head / a.n_kvh, kh = item % a.n_kvh;
    const Item it = resolve_item<MODE>(a, item);
    const uint32_t np = pieces_of(it, ra);
    if (s >= np) return;
    const uint32_t j0 = s * ra.piece, j1 = s + 1u == np ? it.n : j0 + ra.piece;
    const size_t rstride = (size_t)a.n_kvh * ROWB;
    const uint8_t *const kbase = it.kc + (size_t)kh * ROWB, *const vbase = it.vc + (size_t)kh * ROWB;
    const float nsel = c >= 8u ? -1.f : 0.f;

    /* ---- one pass: 16 entries j0 + 16 q + c ---- */
    struct Pass {
        u4_t k[KIND == Q4KV_F16 ? NB : 1];   /* f16 K operands */
        u3_t kw[KIND == Q4KV_Q8 ? NB : 1];   /* q8_0: 12-byte windows */
        uint16_t ks;                         /* scale of block jg of row c */
        u4_t v[KIND == Q4KV_F16 ? 4 : 1];    /* dims U c .. of rows 4 jg + i (U = 8; two dwords for 4) */
        u3_t vw[KIND == Q4KV_Q8 ? 4 : 1];
        uint16_t vs[KIND == Q4KV_Q8 ? 4 : 1];
        uint32_t vmask;                      /* valid entries */
    };
    /* No branch around a load in the loop: past a branch the compiler waits
     * for every outstanding one. Passes past the end re-read the last entry,
     * masked; dense items read a harmless word for theirs. */
    auto entry = [&](uint32_t q) -> int32_t { /* the raw list entry of lane c */
        const uint32_t e = j0 + PASS * q + c, ec = min(e, j1 - 1u);
        if (MODE == MODE_DENSE) return (int32_t)ec;
        return *(const GLOBAL int32_t *)(it.lsrc + (ec & (MODE == MODE_INDEXED ? ~0u : it.lmask)));
    };
    auto issue = [&](uint32_t q, int32_t raw, Pass &p) {
        const uint32_t e = j0 + PASS * q + c;
        const uint32_t m = MODE == MODE_INDEXED ? ~0u : MODE == MODE_DENSE ? 0u : it.lmask;
        const uint32_t at = ((uint32_t)raw & m) | (e & ~m);
        const bool ok = e < j1 && (int32_t)at >= 0 && at < it.max_kv;
        p.vmask = (uint32_t)__ballot(ok) & 0xFFFFu;
        /* padding reads the first valid entry's rows (row 0 without one) */
        const uint32_t first = p.vmask ? __builtin_amdgcn_readlane(at, __builtin_ctz(p.vmask)) : 0u;
        const uint32_t pk = ok ? at : first;
        const uint8_t *kr = kbase + (size_t)pk * rstride;
        if constexpr (KIND == Q4KV_F16) {
#pragma unroll
            for (uint32_t b = 0; b < NB; b++) p.k[b] = ldg((const u4_t *)(kr + 64u * b + 16u * jg));
        } else {
#pragma unroll
            for (uint32_t b = 0; b < NB; b++)
                p.kw[b] = *(const GLOBAL u3u_t *)(kr + 68u * (b >> 1) + 32u * (b & 1u) + 8u * jg);
            p.ks = ldg((const uint16_t *)(kr + 34u * (jg < NB ? jg : 0u)));
        }
        const uint8_t *vr[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
            const uint32_t pv = (uint32_t)__builtin_amdgcn_ds_bpermute((int)((4u * jg + i) * 4u), (int)pk);
            vr[i] = vbase + (size_t)pv * rstride;
        }
        const uint32_t vblk = U * c / 32u;
        if constexpr (KIND == Q4KV_Q8) { /* the scales are looked at first */
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) p.vs[i] = ldg((const uint16_t *)(vr[i] + 34u * vblk));
        }
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
            if constexpr (KIND == Q4KV_F16 && U == 8) {
                p.v[i] = ldg((const u4_t *)(vr[i] + 16u * c));
            } else if constexpr (KIND == Q4KV_F16) {
                const u2_t x = ldg((const u2_t *)(vr[i] + 8u * c));
                p.v[i][0] = x[0];
                p.v[i][1] = x[1];
            } else {
                const uint8_t *w = vr[i] + 68u * (vblk >> 1) + 32u * (vblk & 1u) + (U * c & 31u);
                if constexpr (U == 8) {
                    p.vw[i] = *(const GLOBAL u3u_t *)w;
                } else {
                    const u2_t x = *(const GLOBAL u2u_t *)w;
                    p.vw[i][0] = x[0];
                    p.vw[i][1] = x[1];
                }
            }
        }
    };

    /* an empty cache has no row to stand in */
    const uint32_t nq = it.max_kv ? (j1 - j0 + PASS - 1u) / PASS : 0u;
    Pass pa, pb;
    int32_t e0 = 0, e1 = 0;
    if (nq) {
        e0 = entry(wave);
        e1 = entry(wave + 4u);
    }

    /* ---- Q^T operands: head c mod 8 of each group, dims 32 b + 8 jg ..,
     * q x scale / ln 2 divided by the head's power of two 2^e (its largest
     * magnitude in [0.5, 1)); columns past 7 the residual ---- */
    h8_t qB[HG][NB];
    float qmul[HG];
#pragma unroll
    for (uint32_t k = 0; k < HG; k++) {
        const uint32_t h = 8u * k + (c & 7u);
        const bool hv = h < gqa;
        const float *qr = it.q + (size_t)(hv ? h : 0u) * HD + 8u * jg;
        float x[NB][8], am = 0.f;
#pragma unroll
        for (uint32_t b = 0; b < NB; b++)
#pragma unroll
            for (uint32_t i = 0; i < 8u; i++) x[b][i] = ldg(qr + 32u * b + i);
#pragma unroll
        for (uint32_t b = 0; b < NB; b++)
#pragma unroll
            for (uint32_t i = 0; i < 8u; i++) am = fmaxf(am, fabsf(x[b][i]));
        am = fmaxf(am, __shfl_xor(am, 16));
        am = fmaxf(am, __shfl_xor(am, 32));
        am *= fabsf(a.scale_log2);
        const int e = (am > 0.f && am <= 3.4e38f) ? __builtin_amdgcn_frexp_expf(am) : 0;
        qmul[k] = __builtin_ldexpf(1.f, e);
        const float qs = hv ? __builtin_ldexpf(a.scale_log2, -e) : 0.f;
#pragma unroll
        for (uint32_t b = 0; b < NB; b++)
            qB[k][b] = __builtin_bit_cast(
                h8_t, (u4_t){part_pk(x[b][0] * qs, x[b][1] * qs, nsel), part_pk(x[b][2] * qs, x[b][3] * qs, nsel),
                             part_pk(x[b][4] * qs, x[b][5] * qs, nsel), part_pk(x[b][6] * qs, x[b][7] * qs, nsel)});
    }
    if (nq) issue(wave, e0, pa);

    float m_run[HG], l_run[HG];
    f4_t acc[HG][U];
#pragma unroll
    for (uint32_t k = 0; k < HG; k++) {
        m_run[k] = -INFINITY;
        l_run[k] = 0.f;
#pragma unroll
        for (uint32_t u = 0; u < U; u++) acc[k][u] = (f4_t){0.f, 0.f, 0.f, 0.f};
    }
    VScale vq;
    const uint32_t vodd = (U * c / 32u) & 1u; /* q8_0: this lane's V block is the odd one of its pair */

    auto compute = [&](const Pass &p) {
        f4_t S[HG];
#pragma unroll
        for (uint32_t k = 0; k < HG; k++) S[k] = (f4_t){0.f, 0.f, 0.f, 0.f};
        if constexpr (KIND == Q4KV_F16) {
#pragma unroll
            for (uint32_t b = 0; b < NB; b++)
#pragma unroll
                for (uint32_t k = 0; k < HG; k++)
                    S[k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, p.k[b]), qB[k][b], S[k], 0, 0, 0);
        } else {
            /* the rows' scales, to the lanes that hold their positions */
            if (jg < NB) s_ks[wave][16u * jg + c] = (float)__builtin_bit_cast(_Float16, p.ks);
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (uint32_t b = 0; b < NB; b++) {
                const uint32_t w0 = b & 1u ? p.kw[b][1] : __builtin_amdgcn_alignbyte(p.kw[b][1], p.kw[b][0], 2u);
                const uint32_t w1 = b & 1u ? p.kw[b][2] : __builtin_amdgcn_alignbyte(p.kw[b][2], p.kw[b][1], 2u);
                h2_t x[4];
                biased_h4(w0, x[0], x[1]);
                biased_h4(w1, x[2], x[3]);
                u4_t w;
#pragma unroll
                for (uint32_t i = 0; i < 4u; i++) w[i] = __builtin_bit_cast(uint32_t, x[i] - (h2_t)((_Float16)1152.f));
                const f4_t ks = *(const f4_t *)&s_ks[wave][16u * b + 4u * jg];
#pragma unroll
                for (uint32_t k = 0; k < HG; k++) {
                    const f4_t C = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, w), qB[k][b],
                                                                         (f4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                    for (uint32_t i = 0; i < 4u; i++) S[k][i] = fmaf(ks[i], C[i], S[k][i]);
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
        uint32_t vs[4], vtop = 0u;
        if constexpr (KIND == Q4KV_Q8) {
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) /* a stand-in row may hold inf or NaN */
                vs[i] = (p.vmask >> (4u * jg + i)) & 1u ? p.vs[i] : 0u;
            vtop = max(max(vs[0], vs[1]), max(vs[2], vs[3]));
        }
        h4_t B[HG];
#pragma unroll
        for (uint32_t k = 0; k < HG; k++) {
            float T[4];
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) {
                const float x = add_ror8(S[k][i]) * qmul[k];
                T[i] = (p.vmask >> (4u * jg + i)) & 1u ? x : -INFINITY;
            }
            const float mx = max32(max16(fmax2(fmax2(T[0], T[1]), fmax2(T[2], T[3]))));
            const float mn = fmax2(m_run[k], mx);
            /* one branch for the maximum and for large scales (negative ones,
             * which the quantiser never writes, and infinities come here too) */
            if (__ballot(mn > m_run[k] || (KIND == Q4KV_Q8 && k == 0u && vtop >= 0x6000u)) != 0u) {
                if (KIND == Q4KV_Q8 && k == 0u && !vq.big() &&
                    __ballot(q4kv_big_scale(vs[0]) || q4kv_big_scale(vs[1]) || q4kv_big_scale(vs[2]) ||
                             q4kv_big_scale(vs[3])) != 0u) {
                    vq.divide();
#pragma unroll
                    for (uint32_t h = 0; h < HG; h++)
#pragma unroll
                        for (uint32_t u = 0; u < U; u++) acc[h][u] *= VSCALE_STEP;
                }
                const float alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run[k] - mn);
                l_run[k] *= alpha;
#pragma unroll
                for (uint32_t u = 0; u < U; u++) acc[k][u] *= alpha;
                m_run[k] = mn;
            }
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) T[i] = __builtin_amdgcn_exp2f(T[i] - (mn == -INFINITY ? 0.f : mn));
            l_run[k] += (T[0] + T[1]) + (T[2] + T[3]);
            B[k] = __builtin_bit_cast(h4_t, (u2_t){part_pk(T[0], T[1], nsel), part_pk(T[2], T[3], nsel)});
        }
        /* ---- V, four dims at a time: their values at the lane's four rows
         * [part][row][dim pair], regrouped by dim ---- */
#pragma unroll
        for (uint32_t d = 0; d < U / 4u; d++) {
            uint32_t x[NV][4][2];
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) {
                if constexpr (KIND == Q4KV_F16) {
                    const bool ok = (p.vmask >> (4u * jg + i)) & 1u; /* a stand-in row may hold inf or NaN */
#pragma unroll
                    for (uint32_t e = 0; e < 2u; e++) x[0][i][e] = ok ? p.v[i][2u * d + e] : 0u;
                } else {
                    const h2_t sc = (h2_t)(__builtin_bit_cast(_Float16, (uint16_t)vs[i]));
                    const uint32_t w = __builtin_amdgcn_perm(p.vw[i][d + 1u], p.vw[i][d],
                                                             vodd ? 0x07060504u : 0x05040302u);
                    h2_t y[2];
                    biased_h4(w, y[0], y[1]);
#pragma unroll
                    for (uint32_t e = 0; e < 2u; e++) {
                        const h2_t f = vq.value(y[e]);
                        const h2_t hi = f * sc;
                        x[0][i][e] = __builtin_bit_cast(uint32_t, hi);
                        x[NV - 1u][i][e] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(f, sc, -hi));
                    }
                }
            }
#pragma unroll
            for (uint32_t o = 0; o < 4u; o++) {
                const uint32_t e = o >> 1, sel = o & 1u ? 0x07060302u : 0x05040100u;
#pragma unroll
                for (int v = NV - 1; v >= 0; v--) {
                    const h4_t A = __builtin_bit_cast(h4_t, (u2_t){__builtin_amdgcn_perm(x[v][1][e], x[v][0][e], sel),
                                                                   __builtin_amdgcn_perm(x[v][3][e], x[v][2][e], sel)});
#pragma unroll
                    for (uint32_t k = 0; k < HG; k++)
                        acc[k][4u * d + o] = __builtin_amdgcn_mfma_f32_16x16x16f16(A, B[k], acc[k][4u * d + o], 0, 0, 0);
                }
            }
        }
    };
    for (uint32_t q = wave; q < nq; q += 8u) {
        e0 = entry(q + 8u);
        issue(q + 4u, e1, pb);
        compute(pa);
        e1 = entry(q + 12u);
        issue(q + 8u, e0, pa);
        compute(pb);
    }

    /* ---- merge the waves, then finish or leave the piece's partial ---- */
    const float vmul = vq.undo();
#pragma unroll
    for (uint32_t k = 0; k < HG; k++) {
        const float lw = pair32_sum(sum16(l_run[k]));
        if (lane < 8u) {
            s_m[wave][8u * k + lane] = m_run[k];
            s_l[wave][8u * k + lane] = lw;
        }
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
            float v[U];
#pragma unroll
            for (uint32_t u = 0; u < U; u++) v[u] = add_ror8(acc[k][u][i]) * vmul;
            if (c < 8u) {
                float *d = mrg + (wave * 8u * HG + 8u * k + c) * MROW + U * (4u * jg + i);
#pragma unroll
                for (uint32_t u = 0; u < U; u += 4u) *(f4_t *)(d + u) = (f4_t){v[u], v[u + 1u], v[u + 2u], v[u + 3u]};
            }
        }
    }
    __syncthreads();
    for (uint32_t task = tid; task < gqa * (HD / 4u); task += 256u) {
        const uint32_t g = task / (HD / 4u), d = 4u * (task % (HD / 4u));
        float M = -INFINITY, L = 0.f;
#pragma unroll
        for (uint32_t w = 0; w < 4u; w++) M = fmax2(M, s_m[w][g]);
        f4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (uint32_t w = 0; w < 4u; w++) {
            const float mw = s_m[w][g], f = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M);
            L += f * s_l[w][g];
            v += f * *(const f4_t *)(mrg + (w * 8u * HG + g) * MROW + d);
        }
        if (np == 1u) {
            const float inv = L > 0.f ? 1.f / L : 0.f;
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) {
                float r = v[i] * inv;
                if (it.gate) r *= q4kv_sigmoid(ldg(it.gate + (size_t)g * HD + d + i));
                stg(it.out + (size_t)g * HD + d + i, r);
            }
        } else {
            float *pr = a.part + (((size_t)item * ra.S + s) * gqa + g) * (HD + PHEAD);
            if (d == 0u) stg((fv2 *)pr, (fv2){M, L});
            stg((f4_t *)(pr + PHEAD + d), v);
        }
    }
}

/* Merges the pieces of an (item, head) that has several: HD / 4 lanes of
 * four dims each, NG lane groups with every NG-th piece, eight of them in
 * flight per group. A piece without a valid entry has l = 0; one with l = NaN
 * (scores that are not finite) takes part, as in an item of one piece. */
template <int HD, int MODE> __global__ __launch_bounds__(256) void qsa_rows_merge_k(RowArgs ra) {
    constexpr uint32_t LPH = HD / 4, NG = 256 / LPH;
    __shared__ __attribute__((aligned(16))) f4_t s_acc[256];
    __shared__ float s_m[NG], s_l[NG];
    const AttnArgs &a = ra.a;
    const uint32_t gqa = a.n_head / a.n_kvh, item = a.item0 + blockIdx.y, g = blockIdx.x;
    const uint32_t grp = threadIdx.x / LPH, dl = threadIdx.x % LPH, d = 4u * dl;
    const Item it = resolve_item<MODE>(a, item);
    const uint32_t np = pieces_of(it, ra);
    if (np == 1u) return;
    const float *gp = it.gate ? it.gate + (size_t)g * HD + d : a.part;
    float gt[4];
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) gt[k] = ldg(gp + k);
    const size_t ss = (size_t)gqa * (HD + PHEAD);
    const float *pb = a.part + ((size_t)item * ra.S * gqa + g) * (HD + PHEAD);
    float M = -INFINITY, L = 0.f;
    f4_t acc = {0.f, 0.f, 0.f, 0.f};
    for (uint32_t s0 = grp; s0 < np; s0 += 8u * NG) {
        fv2 ml[8];
        f4_t v[8];
#pragma unroll
        for (uint32_t k = 0; k < 8u; k++) {
            const float *r = pb + (size_t)min(s0 + k * NG, np - 1u) * ss;
            ml[k] = ldg((const fv2 *)r);
            v[k] = ldg((const f4_t *)(r + PHEAD + d));
        }
        float mn = M;
#pragma unroll
        for (uint32_t k = 0; k < 8u; k++)
            if (s0 + k * NG < np && ml[k][1] != 0.f) mn = fmax2(mn, ml[k][0]);
        const float f = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M - mn);
        L *= f;
        acc *= f;
        M = mn;
#pragma unroll
        for (uint32_t k = 0; k < 8u; k++)
            if (s0 + k * NG < np && ml[k][1] != 0.f) {
                const float w = __builtin_amdgcn_exp2f(ml[k][0] - mn);
                L += w * ml[k][1];
                acc += w * v[k];
            }
    }
    s_acc[threadIdx.x] = acc;
    if (dl == 0u) {
        s_m[grp] = M;
        s_l[grp] = L;
    }
    __syncthreads();
    if (grp) return;
    M = -INFINITY;
#pragma unroll
    for (uint32_t k = 0; k < NG; k++) M = fmax2(M, s_m[k]);
    L = 0.f;
    acc = (f4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (uint32_t k = 0; k < NG; k++) {
        const float w = s_m[k] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s_m[k] - M);
        L += w * s_l[k];
        acc += w * s_acc[k * LPH + dl];
    }
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) {
        float r = L != 0.f ? acc[k] / L : 0.f;
        if (it.gate) r *= q4kv_sigmoid(gt[k]);
        stg(it.out + (size_t)g * HD + d + k, r);
    }
}

template <int KIND, int HD, int MODE> void launch(RowArgs ra, uint32_t n_items) {
    const uint32_t gqa = ra.a.n_head / ra.a.n_kvh;
    for (uint32_t i0 = 0; i0 < n_items; i0 += 65535u) {
        const uint32_t ni = std::min(n_items - i0, 65535u);
        ra.a.item0 = i0;
        const bool prof = q4kv_prof_open();
        if (gqa <= 8u)
            qsa_rows_k<KIND, HD, MODE, 1><<<dim3(ra.S, ni), 256, 0, q4kv_stream>>>(ra);
        else
            qsa_rows_k<KIND, HD, MODE, 2><<<dim3(ra.S, ni), 256, 0, q4kv_stream>>>(ra);
        q4kv_prof_close(prof);
        if (ra.S > 1u)
            qsa_rows_merge_k<HD, MODE><<<dim3(gqa, ni), 256, 0, q4kv_stream>>>(ra);
    }
}
template <int KIND, int HD> bool launch_mode(int mode, const RowArgs &ra, uint32_t n_items) {
    if (mode == MODE_DENSE)
        launch<KIND, HD, MODE_DENSE>(ra, n_items);
    else if (mode == MODE_INDEXED)
        launch<KIND, HD, MODE_INDEXED>(ra, n_items);
    else if (mode == MODE_BATCH)
        launch<KIND, HD, MODE_BATCH>(ra, n_items);
    else
        return false;
    return q4kv_launch_ok("qsa rows attention");
}

} // namespace

bool q4kv_rows_takes(int kind, uint32_t hd, uint32_t gqa, bool rows16) {
    if ((kind != Q4KV_Q8 && kind != Q4KV_F16) || (hd != 64u && hd != 128u)) return false;
    static const char *e = getenv("Q4KV_ROWS"); /* 0: the generic kernel (measurement) */
    return gqa <= 16u && rows16 && !(e && e[0] == '0');
}

bool q4kv_rows_launch(int kind, int mode, const AttnArgs &a, uint32_t n_items, uint32_t max_n,
                      float *part, size_t cap) {
    RowArgs ra = {a, 64u, 1u};
    /* The piece: enough of them to fill the 768 workgroups the chip holds
     * (one item of 128 thousand rows: 20 us at 192 entries, 26 at 64, whose
     * starts and partials cost more than they spread), no larger than 192
     * for that, and at most 1/8192 of the longest item times the items: a
     * ragged batch (lengths a third of max_n on average) then still fills
     * the chip several times over (16 sequences: 95 us at 256 entries, 129
     * at 1024). Bounded by a fixed partial capacity, so that every caller's
     * buffer gives the same division. */
    const size_t gqa = a.n_head / a.n_kvh, lim = std::min<size_t>(cap, Q4KV_ROWS_PART);
    const uint64_t total = (uint64_t)max_n * n_items;
    uint64_t piece = std::max<uint64_t>(total / 8192u, std::min<uint64_t>(total / 768u, 192u));
    piece = std::max<uint64_t>(64u, (piece + 63u) / 64u * 64u);
    uint64_t S = (max_n + piece - 1u) / piece;
    if (S < 1u) S = 1u;
    while (S > 1u && (!part || (uint64_t)n_items * S * gqa * (a.hd + PHEAD) > lim)) {
        piece *= 2u;
        S = (max_n + piece - 1u) / piece;
    }
    if (piece > 0x40000000u) piece = 0x40000000u;
    ra.piece = (uint32_t)piece;
    ra.S = (uint32_t)S;
    ra.a.part = part;
    if (kind == Q4KV_Q8)
        return a.hd == 128u ? launch_mode<Q4KV_Q8, 128>(mode, ra, n_items) : launch_mode<Q4KV_Q8, 64>(mode, ra, n_items);
    return a.hd == 128u ? launch_mode<Q4KV_F16, 128>(mode, ra, n_items) : launch_mode<Q4KV_F16, 64>(mode, ra, n_items);
}
