/*
 * q4kv_sparse.hip -- listed attention of many tokens over a q8_0 cache of
 * 256-dim heads: each (token, KV head) item its own position list, up to 16
 * query heads per KV head.
 *
 * Lists of different tokens share few rows, so every item gathers and
 * converts its own; what can be saved is work per row. One workgroup (4
 * waves) per item and split; each wave takes passes of 32 entries and never
 * waits for another one:
 *  - rows go to LDS as 17 sixteen-byte pieces (global_load_lds); K rows of
 *    the next pass are in flight during the softmax and P.V, V rows during
 *    the next scores. Loads straight to registers took 217 us where this
 *    takes 180: their 8- and 16-byte pieces of 16 rows per instruction touch
 *    a row's lines once per block;
 *  - operands are read as aligned dwords, in whatever order of dims they
 *    come: a block pair is 17 dwords; k-group g of K takes dwords 1 + 2 g,
 *    2 + 2 g of the even block and 9 + 2 g, 10 + 2 g of the odd one, lane
 *    k = c mod 4 of V dwords 1 + 4 k .. 4 + 4 k; dword 0 or 8 brings the
 *    scales and the two values that share a dword with one;
 *  - scores S^T = K Q^T (v_mfma_f32_16x16x32_f16) with the exact int8 values
 *    in fp16 and Q^T in two fp16 parts: PACK (up to 8 heads) has the parts in
 *    columns 0-7 and 8-15 of one product, otherwise two products serve up to
 *    16 heads with one conversion of the row; the block scales are applied in
 *    fp32;
 *  - V as v x scale in two fp16 parts, exact (VScale, one for the wave), bytes
 *    of row pairs interleaved by v_perm so that a tile's operand is 8 positions
 *    of one dim: O^T += V^T P^T with no per-head scale work.
 * Tile e, row 4 g + i of the output is dim 64 g + vdim(i, e).
 *
 * What bounds it: the gather (2 x 272 bytes per entry and KV head, three
 * cache lines each) and ~900 VALU instructions per wave and pass, the same
 * for 1 to 16 heads. 512 tokens, 24 / 2 heads, 2051 entries each: 180 us; the
 * slab kernel, which converts every row once per eight heads, 329 us; the
 * gather alone about 130 us.
 */
#include <stdlib.h>
#include <algorithm>

#include "q4kv_attn_item.h"

namespace {

typedef uint32_t u4u_t __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u2u_t __attribute__((ext_vector_type(2), aligned(4)));
typedef float fv2 __attribute__((ext_vector_type(2)));
typedef uint16_t us2 __attribute__((ext_vector_type(2)));

constexpr uint32_t ROWB = 272, PE = 32; /* row bytes, entries per pass */
constexpr uint32_t MROW = 260;          /* merge row: 256 dims, padded */
constexpr float RESCALE = 6.f;
constexpr uint32_t PSTRIDE = 258;       /* split partial: m, l, 256 dims */

/* 16 bytes global -> LDS per lane, in assembly: the compiler would wait for
 * every such DMA before any LDS read (it cannot tell the regions apart); the
 * waits are counted by hand. m0 is a reserved register, its clobber is not
 * honoured: nothing else in this file uses it. */
__device__ inline void dma16(const void *src, void *lds_wave_base) {
    const uint32_t m0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(LOCAL void *)lds_wave_base);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(m0), "v"((const GLOBAL void *)src)
                 : "memory", "m0");
}

/* dim (of a pair's 64) of element e of lane k's V dwords */
__device__ inline uint32_t vdim(uint32_t k, uint32_t e) {
    return k == 0u ? 2u + e : k == 1u ? (e < 14u ? 18u + e : e - 14u) : 16u * k + e;
}
/* dim (of a block's 32) of element i of k-group j's K operand */
__device__ inline uint32_t kdim(uint32_t b, uint32_t j, uint32_t i) {
    if (b & 1u) return 8u * j + i;
    if (j < 3u) return 2u + 8u * j + i;
    return i < 4u ? 26u + i : i < 6u ? i - 4u : 24u + i;
}
__device__ inline uint32_t pk(float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((fv2){x, y}, h2_t));
}
/* bytes 0, 1 (sel 0x04010400) or 2, 3 (0x04030402) of w, biased, as 1024 + u */
__device__ inline h2_t expand(uint32_t w, uint32_t sel) {
    return __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, w, sel));
}

template <bool PACK>
__global__ __launch_bounds__(256, 2) void qsa_sparse_k(AttnArgs a) {
    constexpr uint32_t NH = PACK ? 8 : 16; /* head columns */
    constexpr uint32_t RB = 4u * 2u * PE * ROWB, MB = 4u * NH * MROW * 4u;
    /* each wave's K rows, then V rows; the merge rows take their place */
    __shared__ __attribute__((aligned(16))) uint8_t smem[RB > MB ? RB : MB];
    __shared__ __attribute__((aligned(16))) uint16_t s_ks[4][2][4][4][8]; /* wave, tile, pair, k-group, [even 4 | odd 4] */
    __shared__ u4_t s_ql[PACK ? 1 : 8][PACK ? 1 : 64]; /* Q's second parts (registers would spill) */
    __shared__ float s_m[4][NH], s_l[4][NH];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t c = lane & 15u, jg = lane >> 4, kk = c & 3u;
    uint32_t s, item;
    /* KV heads that share a list on one XCD (their rows are adjacent; xgrp) */
    {
        s = blockIdx.x % a.S;
        const uint32_t L = blockIdx.x / a.S;
        if (a.xgrp) {
            const uint32_t r = L >> 3, t = (r / a.n_kvh) * 8u + (L & 7u);
            if (t >= a.xgrp) return; /* padding of the last group row */
            item = a.item0 + t * a.n_kvh + r % a.n_kvh;
        } else {
            item = a.item0 + L;
        }
    }
    const uint32_t gqa = a.n_head / a.n_kvh, kh = item % a.n_kvh;
    const Item it = resolve_item<MODE_INDEXED>(a, item);
    const bool band = a.band_nb != nullptr;
    const uint32_t n = band ? min((uint32_t)ldg(a.band_nb + item), it.n) : it.n;
    const uint32_t n_all = it.max_kv ? (n + PE - 1u) / PE : 0u;
    const uint32_t q0 = (uint32_t)((uint64_t)n_all * s / a.S), q1 = (uint32_t)((uint64_t)n_all * (s + 1u) / a.S);
    const uint32_t rstride = a.n_kvh * ROWB;
    const uint8_t *const kb = it.kc + (size_t)kh * ROWB, *const vb = it.vc + (size_t)kh * ROWB;
    uint8_t *const kl = smem + wave * 2u * PE * ROWB, *const vl = kl + PE * ROWB;
    const uint8_t *const kr = kl + c * ROWB + 4u + 8u * jg;              /* + 16 tile rows, + 68 pair, + 32 odd */
    const uint8_t *const kx = kl + c * ROWB + (jg == 2u ? 32u : 0u);     /* dword 8 in k-group 2, else 0 */
    const uint8_t *const vr = vl + 4u * jg * ROWB + 68u * (c >> 2) + 4u + 16u * kk;
    const uint8_t *const vx = vl + 4u * jg * ROWB + 68u * (c >> 2) + (kk < 2u ? 0u : 32u);
    const uint32_t ksel = jg == 3u ? 0x05040302u : 0x07060504u;
    const uint32_t vsh = kk < 2u ? 0u : 16u;
    const uint32_t vsel = kk == 1u ? 0x07060100u : 0x03020100u;

    /* ---- the passes' rows: lane l holds the position of entry l mod 32;
     * 17 sixteen-byte pieces per row, nine DMA instructions per cache.
     * Every lane of the first eight and half of the ninth always run, so
     * the counted waits below hold: padding re-reads the first valid
     * entry's row (row 0 without one), passes past the end the last one ---- */
    uint32_t slot[5]; /* DMA slot 64 u + lane: its row x 4 and byte in the row, 16 bits for each u */
#pragma unroll
    for (uint32_t u = 0; u < 10u; u++) {
        const uint32_t x = u * 64u + lane, r = x / 17u;
        const uint32_t w = (r & 31u) * 4u | (x - 17u * r) * 16u << 7;
        slot[u >> 1] = u & 1u ? slot[u >> 1] | w << 16 : w;
    }
    uint32_t pos = 0u, mask_k = 0u;
    auto entry = [&](uint32_t q) { return ldg(it.list + min(PE * q + (lane & 31u), n - 1u)); };
    auto place = [&](uint32_t q, int32_t e) { /* positions and mask of pass q */
        const bool ok = PE * q + (lane & 31u) < n && e >= 0 && (uint32_t)e < it.max_kv;
        mask_k = (uint32_t)__ballot(ok);
        const uint32_t st = mask_k ? (uint32_t)__builtin_amdgcn_readlane(e, __builtin_ctz(mask_k)) : 0u;
        pos = ok ? (uint32_t)e : st;
    };
    auto fetch = [&](const uint8_t *base, uint8_t *dst) {
#pragma unroll
        for (uint32_t u = 0; u < 9u; u++) {
            uint32_t x = slot[u >> 1];
            asm volatile("" : "+v"(x)); /* unpacked here, not ahead of the loop: registers */
            x >>= u & 1u ? 16u : 0u;
            const uint32_t p = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(x & 0x7Fu), (int)pos);
            if (u < 8u || lane < 32u)
                dma16(base + (uint64_t)p * rstride + ((x >> 7) & 0x1FFu), dst + u * 1024u);
        }
    };
    /* The first of this wave's passes q, q + 4, .. that has a valid entry (q1
     * or more: none), eight passes a round trip: a short context's list is
     * padded to the width, and no rows are fetched for that. */
    auto seek = [&](uint32_t q) {
        for (; q < q1; q += 32u) {
            int32_t e[4];
#pragma unroll
            for (uint32_t k = 0; k < 4u; k++) e[k] = entry(q + 8u * k + (lane >> 5) * 4u);
#pragma unroll
            for (uint32_t k = 0; k < 4u; k++) {
                const uint32_t p = q + 8u * k;
                const uint64_t b = __ballot(PE * (p + (lane >> 5) * 4u) + (lane & 31u) < n && e[k] >= 0 &&
                                            (uint32_t)e[k] < it.max_kv);
                if ((uint32_t)b) return p;
                if (b) return p + 4u;
            }
        }
        return q1;
    };
    int32_t e0 = 0;
    uint32_t q = q0 + wave;
    if (q < q1) {
        place(q, entry(q));
        if (!mask_k) {
            q = seek(q + 4u);
            if (q < q1) place(q, entry(q));
        }
        if (q < q1) e0 = entry(q + 4u);
    }

    /* ---- Q^T operands in registers: column c, k-group jg; not for waves that
     * have no pass (padded lists leave most: 64 tokens of 24 / 2 heads at the
     * start of a prompt, 2051 entries, 23.3 us with, 18.7 without) ---- */
    h8_t qh[8];
    float qmul = 1.f;
#pragma unroll
    for (uint32_t b = 0; b < 8u; b++) qh[b] = (h8_t)((_Float16)0.f);
    if (q < q1 || (!PACK && wave == 0u)) {
        const uint32_t h = PACK ? c & 7u : c;
        const bool hv = h < gqa;
        const float *qr = it.q + (size_t)(hv ? h : 0u) * 256u;
        float am = 0.f;
#pragma unroll
        for (uint32_t b = 0; b < 8u; b++)
#pragma unroll
            for (uint32_t i = 0; i < 8u; i++) am = fmaxf(am, fabsf(ldg(qr + 32u * b + 8u * jg + i)));
        am = fmaxf(am, __shfl_xor(am, 16));
        am = fmaxf(am, __shfl_xor(am, 32));
        am *= fabsf(a.scale_log2);
        const int e = (am > 0.f && am <= 3.4e38f) ? __builtin_amdgcn_frexp_expf(am) : 0;
        qmul = __builtin_ldexpf(1.f, e);
        const float qs = hv ? __builtin_ldexpf(a.scale_log2, -e) : 0.f;
#pragma unroll
        for (uint32_t b = 0; b < 8u; b++) {
            u4_t wh, wl;
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) {
                const float y0 = ldg(qr + 32u * b + kdim(b, jg, 2u * i)) * qs;
                const float y1 = ldg(qr + 32u * b + kdim(b, jg, 2u * i + 1u)) * qs;
                wh[i] = pk(y0, y1);
                wl[i] = pk(y0 - h2lo(wh[i]), y1 - h2hi(wh[i]));
                if (PACK && c >= 8u) wh[i] = wl[i];
            }
            qh[b] = __builtin_bit_cast(h8_t, wh);
            if (!PACK && wave == 0u) s_ql[b][lane] = wl;
        }
    }
    /* everything above has landed before the first DMA: a compiler wait for
     * a load would drain the DMAs behind it */
#pragma unroll
    for (uint32_t b = 0; b < 8u; b++) asm volatile("" ::"v"(qh[b]));
    asm volatile("" ::"v"(e0));
    if (!PACK) __syncthreads();
    const float nsel = PACK && c >= 8u ? -1.f : 0.f;
    float m_run = -INFINITY, l_run = 0.f;
    f4_t acc[16];
#pragma unroll
    for (uint32_t e = 0; e < 16u; e++) acc[e] = (f4_t){0.f, 0.f, 0.f, 0.f};

    VScale vq;
    uint32_t mask_v = mask_k;
    if (q < q1) {
        fetch(kb, kl);
        fetch(vb, vl);
    }
    while (q < q1) {
        /* ---- scores, once the K rows have landed (nine V instructions and
         * the list entry may be out) ---- */
        asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
        uint32_t kw[2][4];
#pragma unroll
        for (uint32_t t = 0; t < 2u; t++)
#pragma unroll
            for (uint32_t p = 0; p < 4u; p++) kw[t][p] = *(const uint32_t *)(kx + 16u * ROWB * t + 68u * p);
#pragma unroll
        for (uint32_t t = 0; t < 2u; t++)
#pragma unroll
            for (uint32_t p = 0; p < 4u; p++)
                if (jg >= 2u) /* the odd block's scale in k-group 2, the even one's in 3 */
                    s_ks[wave][t][p][c >> 2][(jg == 2u ? 4u : 0u) + (c & 3u)] =
                        (uint16_t)(jg == 2u ? kw[t][p] >> 16 : kw[t][p]);
        __builtin_amdgcn_wave_barrier();
        f4_t S[2];
        S[0] = S[1] = (f4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (uint32_t p = 0; p < 4u; p++) {
            __builtin_amdgcn_sched_barrier(0); /* operands of one pair at a time: registers */
            h8_t sc[2];
#pragma unroll
            for (uint32_t t = 0; t < 2u; t++) sc[t] = *(const h8_t *)s_ks[wave][t][p][jg];
#pragma unroll
            for (uint32_t o = 0; o < 2u; o++) {
                const uint32_t b = 2u * p + o;
                f4_t C[2];
                h8_t A[2];
#pragma unroll
                for (uint32_t t = 0; t < 2u; t++) {
                    const u2_t x = *(const u2u_t *)(kr + 16u * ROWB * t + 68u * p + 32u * o);
                    uint32_t w0 = x[0], w1 = o ? x[1] : __builtin_amdgcn_perm(x[1], kw[t][p], ksel);
                    w0 ^= 0x80808080u;
                    w1 ^= 0x80808080u;
                    const h2_t bias = (h2_t)((_Float16)1152.f);
                    const h2_t x0 = expand(w0, 0x04010400u) - bias, x1 = expand(w0, 0x04030402u) - bias;
                    const h2_t x2 = expand(w1, 0x04010400u) - bias, x3 = expand(w1, 0x04030402u) - bias;
                    A[t] = (h8_t){x0[0], x0[1], x1[0], x1[1], x2[0], x2[1], x3[0], x3[1]};
                }
                if constexpr (!PACK) {
                    const h8_t ql = __builtin_bit_cast(h8_t, s_ql[b][lane]);
#pragma unroll
                    for (uint32_t t = 0; t < 2u; t++)
                        C[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[t], ql, (f4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                    for (uint32_t t = 0; t < 2u; t++)
                        C[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[t], qh[b], C[t], 0, 0, 0);
                } else {
#pragma unroll
                    for (uint32_t t = 0; t < 2u; t++)
                        C[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[t], qh[b], (f4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                }
#pragma unroll
                for (uint32_t t = 0; t < 2u; t++)
#pragma unroll
                    for (uint32_t i = 0; i < 4u; i++) S[t][i] = fmaf((float)sc[t][4u * o + i], C[t][i], S[t][i]);
            }
        }
        /* the next pass's K rows take the place of this one's: every read of
         * those has returned, and the compiler's wait for the list entry
         * also covers the V rows */
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        mask_v = mask_k;
        q += 4u;
        place(q, e0);
        if (!mask_k && q < q1) {
            q = seek(q + 4u);
            if (q < q1) place(q, entry(q));
        }
        fetch(kb, kl);
        /* ---- softmax (base 2) over the entries of mask_v ---- */
        const uint32_t mask_l = mask_v >> (4u * jg); /* the lane's: bits 0-3 and 16-19 */
        float T[8], mx;
#pragma unroll
        for (uint32_t i = 0; i < 8u; i++) {
            const float x = S[i >> 2][i & 3u];
            T[i] = (PACK ? add_ror8(x) : x) * qmul;
            T[i] = (mask_l >> (i < 4u ? i : i + 12u)) & 1u ? T[i] : -INFINITY;
        }
        mx = fmax2(fmax2(fmax2(T[0], T[1]), fmax2(T[2], T[3])), fmax2(fmax2(T[4], T[5]), fmax2(T[6], T[7])));
        mx = max32(max16(mx));
        /* the running maximum moves when one passes it by RESCALE (the
         * weights then reach 2^RESCALE): a rescale is as long as a softmax */
        if (__ballot(mx > m_run + RESCALE) != 0u) {
            const float mn = fmax2(m_run, mx);
            const float alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run - mn);
            l_run *= alpha;
#pragma unroll
            for (uint32_t e = 0; e < 16u; e++) acc[e] *= alpha;
            m_run = mn;
        }
        const float ms = m_run == -INFINITY ? 0.f : m_run;
        u4_t wh, wl;
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
            const float x0 = __builtin_amdgcn_exp2f(T[2u * i] - ms), x1 = __builtin_amdgcn_exp2f(T[2u * i + 1u] - ms);
            l_run += x0 + x1;
            wh[i] = pk(x0, x1);
            /* PACK: columns past 7 carry the residual instead */
            if constexpr (PACK)
                wh[i] = pk(fmaf(nsel, h2lo(wh[i]), x0), fmaf(nsel, h2hi(wh[i]), x1));
            else
                wl[i] = pk(x0 - h2lo(wh[i]), x1 - h2hi(wh[i]));
        }
        const h8_t Ph = __builtin_bit_cast(h8_t, wh);
        /* ---- V: the lane's eight rows and their scales, in pairs ---- */
        u4_t v4[8];
        uint32_t vw[8];
#pragma unroll
        for (uint32_t r = 0; r < 8u; r++) {
            v4[r] = *(const u4u_t *)(vr + ((r & 3u) + (r & 4u) * 4u) * ROWB);
            vw[r] = *(const uint32_t *)(vx + ((r & 3u) + (r & 4u) * 4u) * ROWB);
        }
        h2_t vs[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
            uint32_t y[2];
#pragma unroll
            for (uint32_t k = 0; k < 2u; k++) {
                const uint32_t r = 2u * i + k;
                y[k] = ((vw[r] >> vsh) & 0xFFFFu) & (uint32_t)__builtin_amdgcn_sbfe((int)mask_l, r < 4u ? r : r + 12u, 1u);
                v4[r][3] = __builtin_amdgcn_perm(vw[r], v4[r][3], vsel);
            }
            vs[i] = __builtin_bit_cast(h2_t, y[0] | y[1] << 16);
        }
        /* large scales (negative ones, which the quantiser never writes, and
         * infinities are looked at too) */
        us2 top = __builtin_bit_cast(us2, vs[0]);
#pragma unroll
        for (uint32_t i = 1; i < 4u; i++) top = __builtin_elementwise_max(top, __builtin_bit_cast(us2, vs[i]));
        if (__ballot(__builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(top, (us2)((uint16_t)0x5FFFu)))) != 0u &&
            !vq.big()) {
            bool b = false;
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) {
                const uint32_t y = __builtin_bit_cast(uint32_t, vs[i]);
                b = b || q4kv_big_scale(y) || q4kv_big_scale(y >> 16);
            }
            if (__ballot(b) != 0u) {
                vq.divide();
#pragma unroll
                for (uint32_t e = 0; e < 16u; e++) acc[e] *= VSCALE_STEP;
            }
        }
        /* ---- O^T += V^T P^T, four dims (one dword per row) at a time ---- */
#pragma unroll
        for (uint32_t d = 0; d < 4u; d++) {
            __builtin_amdgcn_sched_barrier(0);
            uint32_t w[4][2]; /* rows 2 r, 2 r + 1: their bytes 0, 1 / 2, 3 interleaved */
#pragma unroll
            for (uint32_t r = 0; r < 4u; r++) {
                w[r][0] = __builtin_amdgcn_perm(v4[2u * r + 1u][d], v4[2u * r][d], 0x05010400u) ^ 0x80808080u;
                w[r][1] = __builtin_amdgcn_perm(v4[2u * r + 1u][d], v4[2u * r][d], 0x07030602u) ^ 0x80808080u;
            }
#pragma unroll
            for (uint32_t o = 0; o < 4u; o++) {
                u4_t ah, al;
#pragma unroll
                for (uint32_t r = 0; r < 4u; r++) {
                    const h2_t f = vq.value(expand(w[r][o >> 1], o & 1u ? 0x04030402u : 0x04010400u));
                    const h2_t hi = f * vs[r];
                    ah[r] = __builtin_bit_cast(uint32_t, hi);
                    al[r] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(f, vs[r], -hi));
                }
                f4_t &A = acc[4u * d + o];
                A = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, al), Ph, A, 0, 0, 0);
                if constexpr (!PACK)
                    A = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, ah), __builtin_bit_cast(h8_t, wl),
                                                               A, 0, 0, 0);
                A = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, ah), Ph, A, 0, 0, 0);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* V reads returned: refill */
        e0 = entry(q + 4u);
        fetch(vb, vl);
    }

    /* ---- merge the waves ---- */
    const float lw = pair32_sum(sum16(l_run));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); /* the refills past the end */
    __syncthreads(); /* every wave is done with its rows */
    if (lane < NH) {
        s_m[wave][lane] = m_run;
        s_l[wave][lane] = lw;
    }
    float *const mrg = (float *)smem;
    const float vmul = vq.undo();
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++)
#pragma unroll
        for (uint32_t e = 0; e < 16u; e += 2u) {
            fv2 v = {acc[e][i] * vmul, acc[e + 1u][i] * vmul};
            if (PACK) v = (fv2){add_ror8(v[0]), add_ror8(v[1])};
            if (c < NH) *(fv2 *)(mrg + (wave * NH + c) * MROW + 64u * jg + vdim(i, e)) = v;
        }
    __syncthreads();
    for (uint32_t task = tid; task < gqa * 64u; task += 256u) {
        const uint32_t g = task >> 6, d = 4u * (task & 63u);
        float M = -INFINITY, mb = -INFINITY, lb = 0.f;
#pragma unroll
        for (uint32_t w = 0; w < 4u; w++) M = fmax2(M, s_m[w][g]);
        if (band) { /* the band's partial, its rows in out (none: l = 0; l may be NaN) */
            const fv2 ml = ldg((const fv2 *)(a.band_ml + ((size_t)item * gqa + g) * 2u));
            mb = ml[0];
            lb = ml[1];
            if (lb != 0.f) M = fmax2(M, mb);
        }
        float L = 0.f;
        f4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (uint32_t w = 0; w < 4u; w++) {
            const float mw = s_m[w][g], f = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M);
            L += f * s_l[w][g];
            v += f * *(const f4_t *)(mrg + (w * NH + g) * MROW + d);
        }
        float *const o = it.out + (size_t)g * 256u + d;
        if (lb != 0.f) {
            const float f = __builtin_amdgcn_exp2f(mb - M);
            L += f * lb;
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) v[i] += f * ldg(o + i);
        }
        if (a.S == 1u) {
            const float inv = L > 0.f ? 1.f / L : 0.f;
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) {
                float r = v[i] * inv;
                if (it.gate) r *= q4kv_sigmoid(ldg(it.gate + (size_t)g * 256u + d + i));
                stg(o + i, r);
            }
        } else {
            float *pr = a.part + (((size_t)item * a.S + s) * gqa + g) * PSTRIDE;
            if (d == 0u) stg((fv2 *)pr, (fv2){M, L});
            stg((fv2 *)(pr + 2u + d), (fv2){v[0], v[1]});
            stg((fv2 *)(pr + 4u + d), (fv2){v[2], v[3]});
        }
    }
}

} // namespace

bool q4kv_sparse_launch(const AttnArgs &a, uint32_t n_items) {
    const uint32_t gqa = a.n_head / a.n_kvh;
    const uint32_t slots = a.xgrp ? (a.xgrp + 7u) / 8u * 8u * a.n_kvh : n_items;
    if (gqa <= 8u)
        qsa_sparse_k<true><<<slots * a.S, 256, 0, q4kv_stream>>>(a);
    else
        qsa_sparse_k<false><<<slots * a.S, 256, 0, q4kv_stream>>>(a);
    return q4kv_launch_ok("qsa sparse prefill");
}
