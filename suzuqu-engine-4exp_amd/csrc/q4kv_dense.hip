/*
 * q4kv_dense.hip -- dense causal attention of many tokens on gfx950.
 *
 * The dense half of the reference's prefill kernel (gqa_prefill_k,
 * src/q4_rocm.cu:7020-7205): token t of n_tok attends positions
 * 0 .. min(kv_base + t + 1, max_kv) - 1 of a q8_0 or f16 cache,
 *   out = softmax(scale * q.k) v * q4kv_sigmoid(gate).
 *
 * Consecutive tokens see nearly the same positions, so the tokens and the
 * query heads of one KV head are the columns of one matrix product: column
 * r = token * gqa + head, 16 columns per wave, 128 per workgroup. The
 * positions stream through LDS once per workgroup, PT at a time:
 *  - the rows of the next pass are loaded into registers (one cache row
 *    block per thread) while this pass computes, converted once for all 128
 *    columns and stored to the other LDS buffer: one barrier per pass.
 *    q8_0: K as its exact int8 values in fp16 plus the block scales in fp32,
 *    V as v * scale in two fp16 parts, exact (VScale, one for the workgroup);
 *    f16: the rows as stored;
 *  - S^T = K Q^T on v_mfma_f32_16x16x32_f16, Q in two fp16 parts held in
 *    registers (each column's q divided by the power of two that brings its
 *    largest magnitude into [0.5, 1)), the q8_0 block scales applied in fp32
 *    to each block's product;
 *  - online softmax in base 2 per column; the running maximum only moves
 *    when a score exceeds it by more than 2^RESCALE_LOG2, so the
 *    accumulators are rarely rescaled (the weights then reach at most
 *    2^RESCALE_LOG2, far inside fp16);
 *  - O^T += V^T P^T: the weights leave the score tile in the layout the
 *    product needs (slot 8 g + i of a k-group is position 4 g + i, or
 *    16 + 4 g + i - 4 for i >= 4) and are split into two fp16 parts in the
 *    lane; V^T comes from the row-major LDS tile by ds_read_b64_tr_b16.
 * Every contraction keeps ~21 bits of both operands with fp32 accumulation.
 *
 * What bounds it: the matrix pipe. Per (column, position) it issues 2.5
 * (q8_0) or 2 (f16) times the products of the plain fp16 contraction; LDS
 * reads (48 KB per wave and pass at hd 256) stay below the 256 B/clk a CU
 * delivers, and the VALU work per pass (conversion, scales, softmax) is
 * about two thirds of the matrix time and overlaps it across the two waves
 * of a SIMD.
 */
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <math.h>
#include <stdlib.h>
#include <algorithm>
#include <cmath>

#include "q4kv_attn_item.h"

namespace {

typedef short s4_t __attribute__((ext_vector_type(4)));
typedef float f2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u4u_t __attribute__((ext_vector_type(4), aligned(4)));

constexpr uint32_t NWAVE = 8, NTHR = 64 * NWAVE, COLS = 16 * NWAVE;
constexpr float RESCALE_LOG2 = 6.f;
constexpr uint32_t PHEAD = 4; /* a partial row: m, l, two unused floats, HD accumulators */

/* x, y -> two fp16, rounded to nearest (v_cvt_pk_f16_f32) */
__device__ inline uint32_t pk(float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){x, y}, h2_t));
}
/* max of non-NaN operands, without fmaxf's canonicalisations */
__device__ inline float max2(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, INFINITY); }

__device__ inline float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
/* Maximum and sum over the four lanes of a column (16 apart). */
__device__ inline float col_max(float v) {
    v = max2(v, __shfl_xor(v, 16));
    return max2(v, __shfl_xor(v, 32));
}
__device__ inline float col_sum(float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
}

/* Four biased bytes (w ^ 0x80..) -> 1024 + u in four fp16. */
__device__ inline void biased_h4(uint32_t w, h2_t &lo, h2_t &hi) {
    w ^= 0x80808080u;
    lo = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u));
    hi = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u));
}

constexpr uint32_t BAND_MIN = 64;    /* shortest run worth a band */
constexpr uint32_t BAND_SPAN = 1024; /* widest union of a workgroup's bands */
constexpr uint32_t BAND_TOKS = 32;   /* most tokens per workgroup */

/* The band of one token's list (wave-uniform): the run of consecutive
 * positions that ends it (after any padding), at least BAND_MIN long.
 * Returns the list index where the run starts (width if there is none) and
 * the run's first and last positions (ps > pe if none). */
__device__ inline uint32_t band_of(const int32_t *list, uint32_t width, uint32_t max_kv,
                                          uint32_t lane, int32_t &ps, int32_t &pe) {
    ps = 1;
    pe = 0;
    int32_t e = -1, vend = 0;
    for (int32_t base = (int32_t)width - 64;; base -= 64) {
        const int32_t j = base + (int32_t)lane;
        const int32_t v = j >= 0 ? ldg(list + j) : -1;
        const bool ok = j >= 0 && v >= 0 && (uint32_t)v < max_kv;
        const uint64_t bal = __ballot(ok);
        if (bal) {
            const uint32_t hi = 63u - (uint32_t)__builtin_clzll(bal);
            e = base + (int32_t)hi;
            vend = __shfl(v, (int)hi);
            break;
        }
        if (base <= 0) break;
    }
    if (e < 0) return width;
    uint32_t run = 0;
    for (uint32_t w0 = 0; w0 < BAND_SPAN; w0 += 64u) {
        const int32_t j = e - (int32_t)(w0 + lane);
        const bool ok = j >= 0 && ldg(list + j) == vend - (int32_t)(w0 + lane);
        const uint64_t bad = __ballot(!ok);
        if (bad) {
            run = w0 + (uint32_t)__builtin_ctzll(bad);
            break;
        }
        run = w0 + 64u;
    }
    /* a run stops at position 0 (a -1 entry before it equals vend - run too) */
    if ((int64_t)run > (int64_t)vend + 1) run = (uint32_t)vend + 1u;
    if (run > BAND_SPAN) run = BAND_SPAN;
    if (run < BAND_MIN) return width;
    ps = vend - (int32_t)run + 1;
    pe = vend;
    return (uint32_t)(e - (int32_t)run + 1);
}

/* band_of with every load issued at once: the last BAND_NJ x 64 entries of
 * the list (one load per lane each) cover the run whenever the list's last
 * valid entry is among its final 64 (no more than 63 trailing padding or
 * out-of-range entries); otherwise the chained band_of runs. Same result. */
constexpr uint32_t BAND_NJ = BAND_SPAN / 64u + 1u;
__device__ inline uint32_t band_of_tail(const int32_t *list, uint32_t width,
                                               uint32_t max_kv, uint32_t lane, int32_t &ps,
                                               int32_t &pe) {
    int32_t v[BAND_NJ];
#pragma unroll
    for (uint32_t i = 0; i < BAND_NJ; i++) {
        const uint32_t j = 64u * i + lane; /* entry width - 1 - j */
        v[i] = j < width ? ldg(list + (width - 1u - j)) : -1;
    }
    /* the last valid entry: the smallest j with a valid position */
    const uint64_t okb = __ballot(v[0] >= 0 && (uint32_t)v[0] < max_kv);
    if (!okb) return band_of(list, width, max_kv, lane, ps, pe);
    const uint32_t jf = (uint32_t)__builtin_ctzll(okb);
    const int32_t vend = __shfl(v[0], (int)jf);
    /* the run: entry width - 1 - j holds vend - (j - jf) for j = jf, jf + 1, .. */
    uint32_t run = BAND_NJ * 64u - jf; /* every loaded entry from jf on matches */
#pragma unroll
    for (uint32_t i = 0; i < BAND_NJ; i++) {
        const uint32_t j = 64u * i + lane;
        const bool bad = j >= jf && (j >= width || v[i] != vend - (int32_t)(j - jf));
        const uint64_t bb = __ballot(bad);
        if (bb) {
            run = min(run, 64u * i + (uint32_t)__builtin_ctzll(bb) - jf);
            break;
        }
    }
    ps = 1;
    pe = 0;
    /* a run stops at position 0 (a -1 entry before it equals vend - run too) */
    if ((int64_t)run > (int64_t)vend + 1) run = (uint32_t)vend + 1u;
    if (run > BAND_SPAN) run = BAND_SPAN;
    if (run < BAND_MIN) return width;
    ps = vend - (int32_t)run + 1;
    pe = vend;
    return width - 1u - jf - run + 1u;
}

struct Args {
    const uint8_t *kc, *vc;
    const float *q, *gate;
    float *out, *part;
    uint32_t n_head, n_kvh, gqa, n_tok, kv_base, max_kv, n_tiles;
    /* tiles from T1 on run in S splits of their positions; dispatch order:
     * the unsplit tiles T1 - 1 .. T2, the split ones, the tiles below T2 */
    uint32_t S, T1, T2;
    float scale_log2;
    /* the band form (qsa_dense_k with BAND): lists, tokens per tile, and per
     * item the entries before its band and the band's (m, l) per head */
    const int32_t *idx;
    uint64_t tok_stride, kvh_stride;
    uint32_t width, toks;
    int32_t *band_nb;
    float *band_ml;
};

/* One pass's tile geometry. 256 threads hold one 32-value q8_0 block of K
 * (the other 256 of V) each, so PT x HD = 8192 values per pass. */
template <int KIND, int HD> struct Geo {
    static constexpr uint32_t NB = HD / 32, PT = 8192 / HD, NT = PT / 16, KG = PT / 32;
    static constexpr uint32_t KS = HD * 2 + 32; /* K row bytes in LDS (conflict-free 16-row reads: 4.4 cycles against 8 with 16 bytes of padding) */
    static constexpr uint32_t VS = HD * 2;      /* V row bytes (swizzled, see vaddr) */
    static constexpr uint32_t NV = KIND == Q4KV_Q8 ? 2 : 1; /* V parts */
    static constexpr uint32_t ROWB = KIND == Q4KV_Q8 ? NB * 34 : HD * 2;
};

/* Byte offset of the 16-byte piece `pc` of V row p. The transposing read of
 * 16 dims takes 32 bytes of each of 8 rows per half wave: rows are rotated
 * by 32-byte windows (xor p mod 8 over 8 windows), which puts them on
 * distinct banks; the two pieces of a window trade places every 8 rows so
 * that the conversion's stores (16 rows of one piece) are conflict-free
 * too. A row of 128 bytes holds four windows, two rows cover the banks. */
template <uint32_t VS> __device__ inline uint32_t vaddr(uint32_t p, uint32_t pc) {
    const uint32_t x = VS >= 256 ? p & 7u : (p >> 1) & 3u;
    return p * VS + (((pc >> 1) ^ x) << 5) + (((pc ^ (p >> 3)) & 1u) << 4);
}

/* BAND: listed prefill's shared part. A token's band is the longest run of
 * consecutive positions that ends its list (the causal recent window, which
 * consecutive tokens share); the tile's columns then see the positions of
 * their own bands only, out of the union of the tile's bands, and leave
 * (m, l) and unnormalised rows (in out) for the kernel that attends the list
 * entries before the bands. A tile is whole tokens. Without a band for some
 * token, or with a union past BAND_SPAN, the list is left as it is. */
template <int KIND, int HD, bool BAND = false>
__global__ __launch_bounds__(512, 2) void qsa_dense_k(Args a) {
    using G = Geo<KIND, HD>;
    constexpr uint32_t NB = G::NB, PT = G::PT, NT = G::NT, KG = G::KG, KS = G::KS, VS = G::VS;
    constexpr uint32_t TD = HD / 16; /* output tiles of 16 dims */
    __shared__ __attribute__((aligned(16))) uint8_t s_k[2][PT * KS];
    __shared__ __attribute__((aligned(16))) uint8_t s_v[2][G::NV][PT * VS];
    /* K block scales, in the order the score stages read them: [tile pair]
     * [block][k-group][tile][position], 16 bytes per lane and stage */
    __shared__ __attribute__((aligned(16))) uint16_t s_ks[KIND == Q4KV_Q8 ? 2 : 1][KIND == Q4KV_Q8 ? NB * PT : 8];
    /* 1 + the last pass whose V rows hold a value that is not finite; 1 + the
     * last one with a V scale that VScale divides for (mod 2^16: what either
     * leads to is right, if not needed, at any pass) */
    __shared__ __attribute__((aligned(4))) uint16_t s_flag[2][2];
    __shared__ uint32_t s_nan[PT * NB]; /* a pass's values that are not finite, one bit each */

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t c = lane & 15u, jg = lane >> 4;
    /* longest pieces first: the grid drains evenly */
    uint32_t s = 0u, S = 1u, tile, kh = blockIdx.x;
    const uint32_t mid = (a.T1 - a.T2) * a.n_kvh, hi = mid + (a.n_tiles - a.T1) * a.S * a.n_kvh;
    if (kh < mid) {
        tile = a.T1 - 1u - kh / a.n_kvh;
    } else if (kh < hi) {
        kh -= mid;
        S = a.S;
        s = kh % S;
        kh /= S;
        tile = a.n_tiles - 1u - kh / a.n_kvh;
    } else {
        kh -= hi;
        tile = a.T2 - 1u - kh / a.n_kvh;
    }
    kh %= a.n_kvh;
    const uint32_t gqa = a.gqa;
    /* this lane's column */
    const uint32_t lc = wave * 16u + c, col = tile * COLS + lc;
    const uint32_t t_in = BAND ? lc / gqa : 0u;
    const bool live = BAND ? t_in < a.toks && tile * a.toks + t_in < a.n_tok : col < a.n_tok * gqa;
    const uint32_t t = !live ? 0u : BAND ? tile * a.toks + t_in : col / gqa;
    const uint32_t h = !live ? 0u : BAND ? lc - t_in * gqa : col - t * gqa;
    /* the column sees positions lo_c .. n_c - 1, the workgroup's columns
     * together lo_all .. n_all - 1, and all of them lo_max .. n_min - 1 */
    uint32_t lo_c = 0u, n_c, lo_all = 0u, n_all, lo_max = 0u, n_min;
    if constexpr (BAND) {
        __shared__ int32_t s_lo[BAND_TOKS], s_hi[BAND_TOKS]; /* first and last position, hi < lo: none */
        __shared__ uint32_t s_nb[BAND_TOKS];
        for (uint32_t k = wave; k < a.toks; k += NWAVE) {
            const uint32_t tk = tile * a.toks + k;
            int32_t ps = 1, pe = 0;
            uint32_t nb = a.width;
            if (tk < a.n_tok)
                nb = band_of_tail(a.idx + (size_t)tk * a.tok_stride + (size_t)kh * a.kvh_stride, a.width,
                                  a.max_kv, lane, ps, pe);
            if (lane == 0u) {
                s_lo[k] = ps;
                s_hi[k] = pe;
                s_nb[k] = nb;
            }
        }
        __syncthreads();
        /* over the tile's tokens, one per lane: one after the other, with LDS
         * round trips each, 32 tokens took 2.5 us, a tenth of a launch over
         * short lists (100 tokens, 32 / 8 heads, 150 entries: 39.5 us, now 37.0) */
        int32_t lo = INT32_MAX, hi = INT32_MIN, lom = 0, him = INT32_MAX;
        {
            const uint32_t k = lane % BAND_TOKS;
            if (k < a.toks && tile * a.toks + k < a.n_tok) {
                const int32_t l = s_lo[k], h = s_hi[k];
                const bool has = l <= h;
                lo = has ? l : lo;
                hi = has ? h : hi;
                lom = has ? l : 0;
                him = has ? h : -1;
            }
#pragma unroll
            for (int d = 1; d < (int)BAND_TOKS; d *= 2) {
                lo = min(lo, __shfl_xor(lo, d));
                hi = max(hi, __shfl_xor(hi, d));
                lom = max(lom, __shfl_xor(lom, d));
                him = min(him, __shfl_xor(him, d));
            }
            lo = __builtin_amdgcn_readfirstlane(lo);
            hi = __builtin_amdgcn_readfirstlane(hi);
            lom = __builtin_amdgcn_readfirstlane(lom);
            him = __builtin_amdgcn_readfirstlane(him);
        }
        const bool use = lo <= hi && (int64_t)hi - lo + 1 <= (int64_t)BAND_SPAN;
        if (tid < a.toks && tile * a.toks + tid < a.n_tok) {
            const uint32_t item = (tile * a.toks + tid) * a.n_kvh + kh;
            a.band_nb[item] = (int32_t)(use ? s_nb[tid] : a.width);
            if (!use || s_lo[tid] > s_hi[tid])
                for (uint32_t g = 0; g < gqa; g++)
                    stg((f2_t *)(a.band_ml + ((size_t)item * gqa + g) * 2u), (f2_t){-INFINITY, 0.f});
        }
        if (!use) return; /* uniform over the workgroup */
        lo_all = (uint32_t)lo;
        n_all = (uint32_t)hi + 1u;
        lo_max = (uint32_t)lom;
        n_min = (uint32_t)(him + 1);
        lo_c = live ? (uint32_t)s_lo[t_in] : 0u;
        n_c = live ? (uint32_t)(s_hi[t_in] + 1) : 0u; /* none: 1 .. 0, nothing */
    } else {
        auto seen = [&](uint32_t tok) { /* positions token tok attends */
            const uint64_t n = (uint64_t)a.kv_base + tok + 1u;
            return n < a.max_kv ? (uint32_t)n : a.max_kv;
        };
        n_c = live ? seen(t) : 0u;
        const uint32_t c_last = min((tile + 1u) * COLS, a.n_tok * gqa) - 1u;
        n_all = seen(c_last / gqa);       /* of the workgroup's last token */
        n_min = seen(tile * COLS / gqa);  /* of its first */
    }
    auto sees = [&](uint32_t p) { return p < n_c && (!BAND || p >= lo_c); };
    auto partly = [&](uint32_t base) { /* some column does not see all of the pass */
        return base + PT > n_min || (BAND && base < lo_max);
    };
    const uint32_t n_pass = (n_all - lo_all + PT - 1u) / PT;
    const uint32_t p0 = (uint32_t)((uint64_t)n_pass * s / S);
    const uint32_t p1 = (uint32_t)((uint64_t)n_pass * (s + 1u) / S);
    if (tid < 4u) s_flag[tid >> 1][tid & 1u] = 0u;
    VScale vq;

    /* ---- this thread's share of a pass's rows ---- */
    const size_t rstride = (size_t)a.n_kvh * G::ROWB;
    const uint8_t *const kb = a.kc + (size_t)kh * G::ROWB, *const vb = a.vc + (size_t)kh * G::ROWB;
    /* q8_0: threads 0-255 one K block, 256-511 one V block; 16 rows x 4
     * blocks per wave */
    const bool is_v = wave >= NWAVE / 2u;
    const uint32_t u = tid & 255u;
    const uint32_t bp = (u & 15u) + 16u * (u / (16u * NB)), bb = (u >> 4) % NB;
    const uint32_t bsel = bb & 1u ? 0x07060504u : 0x05040302u; /* block bytes of two dwords */
    u4_t r0, r1;
    uint32_t r2;
    u4_t rk[2], rv[2]; /* f16 */
    auto load = [&](uint32_t pass) {
        if constexpr (KIND == Q4KV_Q8) {
            const uint32_t p = min(lo_all + pass * PT + bp, n_all - 1u);
            const uint8_t *src = (is_v ? vb : kb) + (size_t)p * rstride + 68u * (bb >> 1) + 32u * (bb & 1u);
            r0 = *(const GLOBAL u4u_t *)src;
            r1 = *(const GLOBAL u4u_t *)(src + 16);
            r2 = ldg((const uint32_t *)(src + 32));
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 2u; i++) {
                const uint32_t e = tid + NTHR * i, pc = e % (HD / 8u);
                const uint32_t p = min(lo_all + pass * PT + e / (HD / 8u), n_all - 1u);
                rk[i] = ldg((const u4_t *)(kb + (size_t)p * rstride) + pc);
                rv[i] = ldg((const u4_t *)(vb + (size_t)p * rstride) + pc);
            }
        }
    };
    auto store = [&](uint32_t pass) {
        const uint32_t buf = pass & 1u;
        const bool masked = partly(lo_all + pass * PT);
        if constexpr (KIND == Q4KV_Q8) {
            const uint32_t d[9] = {r0[0], r0[1], r0[2], r0[3], r1[0], r1[1], r1[2], r1[3], r2};
            /* even blocks: the scale leads the first dword; odd blocks: it
             * ends it */
            const uint16_t sb = (uint16_t)(bb & 1u ? d[0] >> 16 : d[0]);
            if (!is_v) {
                uint8_t *dst = s_k[buf] + bp * KS + 64u * bb;
#pragma unroll
                for (uint32_t k = 0; k < 4u; k++) {
                    h2_t x[4];
                    biased_h4(__builtin_amdgcn_perm(d[2u * k + 1u], d[2u * k], bsel), x[0], x[1]);
                    biased_h4(__builtin_amdgcn_perm(d[2u * k + 2u], d[2u * k + 1u], bsel), x[2], x[3]);
                    u4_t w;
#pragma unroll
                    for (uint32_t i = 0; i < 4u; i++)
                        w[i] = __builtin_bit_cast(uint32_t, x[i] - (h2_t)((_Float16)1152.f));
                    *(u4_t *)(dst + 16u * k) = w;
                }
                s_ks[buf][(((bp >> 5) * NB + bb) * 4u + ((bp >> 2) & 3u)) * 8u + ((bp >> 4) & 1u) * 4u +
                          (bp & 3u)] = sb;
            } else {
                const h2_t vs = (h2_t)(__builtin_bit_cast(_Float16, sb));
#pragma unroll
                for (uint32_t k = 0; k < 4u; k++) {
                    h2_t x[4];
                    biased_h4(__builtin_amdgcn_perm(d[2u * k + 1u], d[2u * k], bsel), x[0], x[1]);
                    biased_h4(__builtin_amdgcn_perm(d[2u * k + 2u], d[2u * k + 1u], bsel), x[2], x[3]);
                    u4_t wh, wl;
#pragma unroll
                    for (uint32_t i = 0; i < 4u; i++) {
                        /* v, exact; its product with the scale rounded once,
                         * and what the rounding left */
                        const h2_t f = vq.value(x[i]);
                        const h2_t hi = f * vs;
                        wh[i] = __builtin_bit_cast(uint32_t, hi);
                        wl[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(f, vs, -hi));
                    }
                    const uint32_t at = vaddr<VS>(bp, 4u * bb + k);
                    *(u4_t *)(s_v[buf][0] + at) = wh;
                    *(u4_t *)(s_v[buf][G::NV - 1u] + at) = wl;
                }
                if (masked && (sb & 0x7C00u) == 0x7C00u) s_flag[buf][0] = (uint16_t)(pass + 1u);
                if (q4kv_big_scale(sb)) s_flag[buf][1] = (uint16_t)(pass + 1u);
            }
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 2u; i++) {
                const uint32_t e = tid + NTHR * i, pc = e % (HD / 8u), p = e / (HD / 8u);
                *(u4_t *)(s_k[buf] + p * KS + 16u * pc) = rk[i];
                *(u4_t *)(s_v[buf][0] + vaddr<VS>(p, pc)) = rv[i];
                if (masked) {
                    bool bad = false;
#pragma unroll
                    for (uint32_t k = 0; k < 4u; k++)
                        bad = bad || (rv[i][k] & 0x7C00u) == 0x7C00u ||
                              (rv[i][k] & 0x7C000000u) == 0x7C000000u;
                    if (bad) s_flag[buf][0] = (uint16_t)(pass + 1u);
                }
            }
        }
    };
    if (p0 < p1) load(p0);

    /* ---- this wave's Q^T operands: column c, dims 32 b + 8 jg .. + 7, q x
     * scale / ln 2 divided by the column's power of two 2^e, in two parts ---- */
    h8_t qh[NB], ql[NB];
    float qmul;
    {
        const float *qr = a.q + ((size_t)t * a.n_head + kh * gqa + h) * HD + 8u * jg;
        const bool al = ((uintptr_t)a.q & 15u) == 0u;
        float x[NB][8];
#pragma unroll
        for (uint32_t b = 0; b < NB; b++) {
            if (al) {
                const f4_t x0 = ldg((const f4_t *)(qr + 32u * b)), x1 = ldg((const f4_t *)(qr + 32u * b + 4u));
#pragma unroll
                for (uint32_t i = 0; i < 4u; i++) {
                    x[b][i] = x0[i];
                    x[b][4u + i] = x1[i];
                }
            } else {
#pragma unroll
                for (uint32_t i = 0; i < 8u; i++) x[b][i] = ldg(qr + 32u * b + i);
            }
        }
        float am = 0.f;
#pragma unroll
        for (uint32_t b = 0; b < NB; b++)
#pragma unroll
            for (uint32_t i = 0; i < 8u; i++) am = fmaxf(am, fabsf(x[b][i]));
        am = fmaxf(am, __shfl_xor(am, 16));
        am = fmaxf(am, __shfl_xor(am, 32));
        am *= fabsf(a.scale_log2);
        const int e = (am > 0.f && am <= 3.4e38f) ? __builtin_amdgcn_frexp_expf(am) : 0;
        qmul = __builtin_ldexpf(1.f, e);
        const float qs = live ? __builtin_ldexpf(a.scale_log2, -e) : 0.f;
#pragma unroll
        for (uint32_t b = 0; b < NB; b++) {
            u4_t wh, wl;
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) {
                const float y0 = x[b][2u * i] * qs, y1 = x[b][2u * i + 1u] * qs;
                wh[i] = pk(y0, y1);
                wl[i] = pk(y0 - h2lo(wh[i]), y1 - h2hi(wh[i]));
            }
            qh[b] = __builtin_bit_cast(h8_t, wh);
            ql[b] = __builtin_bit_cast(h8_t, wl);
        }
    }

    float m_run = -INFINITY, l_run = 0.f;
    uint64_t nan_out = 0u; /* bit 4 T + i: acc[T][i] sums a value that is not finite */
    f4_t acc[TD];
#pragma unroll
    for (uint32_t T = 0; T < TD; T++) acc[T] = (f4_t){0.f, 0.f, 0.f, 0.f};

    __syncthreads(); /* s_flag cleared */
    if (p0 < p1) store(p0);
    __syncthreads();

    for (uint32_t pass = p0; pass < p1; pass++) {
        const uint32_t buf = pass & 1u, base = lo_all + pass * PT;
        const bool masked = partly(base);
        const uint32_t flag_at = *(const uint32_t *)s_flag[buf];
        if (pass + 1u < p1) load(pass + 1u);
        /* ---- scores: tile tt holds positions base + 16 tt + 4 jg + i of
         * column c. Eight stages of two tiles and one block; the operands of
         * the stage after next are in flight, and the scales are applied one
         * stage late ---- */
        f4_t S[NT], Sl[KIND == Q4KV_Q8 ? 1 : NT];
#pragma unroll
        for (uint32_t tt = 0; tt < NT; tt++) S[tt] = (f4_t){0.f, 0.f, 0.f, 0.f};
        if constexpr (KIND != Q4KV_Q8) {
#pragma unroll
            for (uint32_t tt = 0; tt < NT; tt++) Sl[tt] = (f4_t){0.f, 0.f, 0.f, 0.f};
        }
        {
            const uint8_t *kr = s_k[buf] + c * KS + 16u * jg;
            const uint16_t *ksr = s_ks[KIND == Q4KV_Q8 ? buf : 0u] + 8u * jg;
            h8_t A[8][2], ks[8];
            auto fetch = [&](uint32_t st) {
                const uint32_t b = st % NB, tp = st / NB;
#pragma unroll
                for (uint32_t k = 0; k < 2u; k++)
                    A[st][k] = *(const h8_t *)(kr + (2u * tp + k) * 16u * KS + 64u * b);
                if constexpr (KIND == Q4KV_Q8) ks[st] = *(const h8_t *)(ksr + st * 32u);
            };
            f4_t C[8][2];
            auto scale = [&](uint32_t st) {
                const uint32_t tp = st / NB;
#pragma unroll
                for (uint32_t k = 0; k < 2u; k++)
#pragma unroll
                    for (uint32_t i = 0; i < 4u; i++)
                        S[2u * tp + k][i] = fmaf((float)ks[st][4u * k + i], C[st][k][i], S[2u * tp + k][i]);
            };
            fetch(0u);
            fetch(1u);
#pragma unroll
            for (uint32_t st = 0; st < 8u; st++) {
                const uint32_t b = st % NB, tp = st / NB;
                if (st + 2u < 8u) fetch(st + 2u);
                if constexpr (KIND == Q4KV_Q8) {
#pragma unroll
                    for (uint32_t k = 0; k < 2u; k++)
                        C[st][k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[st][k], ql[b], (f4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                    for (uint32_t k = 0; k < 2u; k++)
                        C[st][k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[st][k], qh[b], C[st][k], 0, 0, 0);
                    if (st) scale(st - 1u);
                } else {
#pragma unroll
                    for (uint32_t k = 0; k < 2u; k++)
                        Sl[2u * tp + k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[st][k], ql[b], Sl[2u * tp + k], 0, 0, 0);
#pragma unroll
                    for (uint32_t k = 0; k < 2u; k++)
                        S[2u * tp + k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[st][k], qh[b], S[2u * tp + k], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (KIND == Q4KV_Q8) {
                scale(7u);
            } else {
                /* the small parts summed apart: half the roundings at the
                 * sum's magnitude */
#pragma unroll
                for (uint32_t tt = 0; tt < NT; tt++) S[tt] += Sl[tt];
            }
        }
        /* ---- V^T operands of the first product stage, ahead of the softmax;
         * a stage is two tiles of 16 dims over one k-group of 32 positions ---- */
        h8_t VA[8][2][G::NV];
        const uint32_t at0 = vaddr<VS>(4u * jg + (c >> 2), (c >> 1) & 1u) + 8u * (c & 1u);
        auto vfetch = [&](uint32_t st) {
            const uint32_t kg = st / (TD / 2u), T0 = 2u * (st % (TD / 2u));
#pragma unroll
            for (uint32_t k = 0; k < 2u; k++) {
                /* vaddr(row, 2 T + ..): T enters by the window's xor */
                const uint32_t at = (at0 ^ ((T0 + k) << 5)) + kg * 32u * VS;
#pragma unroll
                for (uint32_t v = 0; v < G::NV; v++) {
                    const s4_t a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LOCAL s4_t *)(s_v[buf][v] + at));
                    const s4_t a1 =
                        __builtin_amdgcn_ds_read_tr16_b64_v4i16((LOCAL s4_t *)(s_v[buf][v] + at + 16u * VS));
                    VA[st][k][v] = __builtin_bit_cast(h8_t, __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7));
                }
            }
        };
        vfetch(0u);
        /* ---- online softmax (base 2) ---- */
        if (masked) {
#pragma unroll
            for (uint32_t tt = 0; tt < NT; tt++)
#pragma unroll
                for (uint32_t i = 0; i < 4u; i++)
                    S[tt][i] = sees(base + 16u * tt + 4u * jg + i) ? S[tt][i] : -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (uint32_t tt = 0; tt < NT; tt++) mx = max3(max3(mx, S[tt][0], S[tt][1]), S[tt][2], S[tt][3]);
        mx *= qmul;
        /* this lane's positions only: the column's maximum is formed when a
         * lane passes the limit */
        const uint32_t flag = __builtin_amdgcn_readfirstlane(flag_at);
        const bool bad = masked && (flag & 0xFFFFu) == ((pass + 1u) & 0xFFFFu);
        const bool grow = KIND == Q4KV_Q8 && !vq.big() && flag >> 16 == ((pass + 1u) & 0xFFFFu);
        const bool up = __ballot(mx > m_run + RESCALE_LOG2) != 0u;
        if (up || bad || grow) {
            if (bad || grow) { /* the whole workgroup */
                __syncthreads();
                if (grow) {
                    /* V over 128 from this pass on: its rows once more */
                    vq.divide();
#pragma unroll
                    for (uint32_t T = 0; T < TD; T++) acc[T] *= VSCALE_STEP;
#pragma unroll 1
                    for (uint32_t i = tid; i < PT * (HD / 8u); i += NTHR) {
                        const uint32_t p = i / (HD / 8u), pc = i % (HD / 8u), b = pc / 4u;
                        const uint8_t *blk = vb + (size_t)min(base + p, n_all - 1u) * rstride + 34u * b;
                        const h2_t vs = (h2_t)(__builtin_bit_cast(_Float16, ldg((const uint16_t *)blk)));
                        u4_t wh, wl;
#pragma unroll
                        for (uint32_t e = 0; e < 4u; e++) {
                            const uint32_t w = ldg((const uint16_t *)(blk + 2u + 8u * (pc & 3u)) + e) ^ 0x8080u;
                            const h2_t f = vq.value(__builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u)));
                            const h2_t hi = f * vs;
                            wh[e] = __builtin_bit_cast(uint32_t, hi);
                            wl[e] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(f, vs, -hi));
                        }
                        *(u4_t *)(s_v[buf][0] + vaddr<VS>(p, pc)) = wh;
                        *(u4_t *)(s_v[buf][G::NV - 1u] + vaddr<VS>(p, pc)) = wl;
                    }
                    __syncthreads();
                }
                if (bad) {
                    /* Rows that not every column sees hold inf or NaN, which a zero
                     * weight would turn into NaN. They are taken out of the tile,
                     * and the outputs of the columns that do see them become NaN
                     * at the end (as inf x weight parts gives in every kernel). */
                    for (uint32_t i = tid; i < PT * NB; i += NTHR) s_nan[i] = 0u;
                    __syncthreads();
                    for (uint32_t i = tid; i < PT * (HD / 8u); i += NTHR) {
                        const uint32_t p = i / (HD / 8u), pc = i % (HD / 8u), at = vaddr<VS>(p, pc);
                        uint32_t bits = 0u;
                        for (uint32_t e = 0; e < 8u; e++) {
                            uint16_t *v = (uint16_t *)(s_v[buf][0] + at) + e;
                            if ((*v & 0x7C00u) != 0x7C00u) continue;
                            bits |= 1u << e;
                            *v = 0u;
                            if (G::NV == 2) ((uint16_t *)(s_v[buf][G::NV - 1u] + at))[e] = 0u;
                        }
                        if (bits) atomicOr(&s_nan[p * NB + pc / 4u], bits << (8u * (pc & 3u)));
                    }
                    __syncthreads();
                    for (uint32_t p = 0; p < PT && base + p < n_c; p++)
                        for (uint32_t b = 0; b < NB && sees(base + p); b++) {
                            const uint32_t w = s_nan[p * NB + b] >> (4u * jg);
                            nan_out |= ((uint64_t)(w & 15u) | (uint64_t)((w >> 16) & 15u) << 4) << (8u * b);
                        }
                }
                __syncthreads();
                vfetch(0u);
            }
            if (up) {
                const float mn = max2(m_run, col_max(mx));
                const float alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run - mn);
                m_run = mn;
                l_run *= alpha;
#pragma unroll
                for (uint32_t T = 0; T < TD; T++) acc[T] *= alpha;
            }
        }
        const float ms = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
        for (uint32_t tt = 0; tt < NT; tt++) {
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) S[tt][i] = __builtin_amdgcn_exp2f(fmaf(S[tt][i], qmul, -ms));
            l_run += (S[tt][0] + S[tt][1]) + (S[tt][2] + S[tt][3]);
        }
        /* ---- O^T += V^T P^T ---- */
        h8_t Ph[KG], Pl[KG];
#pragma unroll
        for (uint32_t kg = 0; kg < KG; kg++) {
            u4_t wh, wl;
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) {
                const f4_t &P = S[2u * kg + (i >> 1)];
                const float x0 = P[2u * (i & 1u)], x1 = P[2u * (i & 1u) + 1u];
                wh[i] = pk(x0, x1);
                wl[i] = pk(x0 - h2lo(wh[i]), x1 - h2hi(wh[i]));
            }
            Ph[kg] = __builtin_bit_cast(h8_t, wh);
            Pl[kg] = __builtin_bit_cast(h8_t, wl);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t st = 0; st < 8u; st++) {
            const uint32_t kg = st / (TD / 2u), T0 = 2u * (st % (TD / 2u));
            if (st + 1u < 8u) vfetch(st + 1u);
            if constexpr (G::NV == 2) {
#pragma unroll
                for (uint32_t k = 0; k < 2u; k++)
                    acc[T0 + k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(VA[st][k][1], Ph[kg], acc[T0 + k], 0, 0, 0);
            }
#pragma unroll
            for (uint32_t k = 0; k < 2u; k++)
                acc[T0 + k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(VA[st][k][0], Pl[kg], acc[T0 + k], 0, 0, 0);
#pragma unroll
            for (uint32_t k = 0; k < 2u; k++)
                acc[T0 + k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(VA[st][k][0], Ph[kg], acc[T0 + k], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (pass + 1u < p1) store(pass + 1u);
        __syncthreads();
    }

    /* ---- the columns' rows: finished, or the split's partial ---- */
    const float l = col_sum(l_run);
    if (!live) return;
    if (nan_out) {
#pragma unroll
        for (uint32_t T = 0; T < TD; T++)
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++)
                if ((nan_out >> (4u * T + i)) & 1u) acc[T][i] = __builtin_nanf("");
    }
    const float vmul = vq.undo();
    if constexpr (BAND) {
        if (lo_c >= n_c) return; /* no band: written above */
        const size_t item = (size_t)t * a.n_kvh + kh;
        if (jg == 0u) stg((f2_t *)(a.band_ml + (item * gqa + h) * 2u), (f2_t){m_run, l});
        float *o = a.out + ((size_t)t * a.n_head + kh * gqa + h) * HD + 4u * jg;
#pragma unroll
        for (uint32_t T = 0; T < TD; T++)
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) stg(o + 16u * T + i, acc[T][i] * vmul);
        return;
    }
    if (S > 1u) {
        const uint32_t c_hi = a.n_tok * gqa - a.T1 * COLS; /* split columns per KV head */
        float *pb = a.part + (((size_t)kh * c_hi + (col - a.T1 * COLS)) * S + s) * (HD + PHEAD);
        if (jg == 0u) stg((f2_t *)pb, (f2_t){m_run, l});
#pragma unroll
        for (uint32_t T = 0; T < TD; T++) stg((f4_t *)(pb + PHEAD + 16u * T + 4u * jg), acc[T] * vmul);
        return;
    }
    const float inv = l > 0.f ? vmul / l : 0.f;
    const size_t ro = ((size_t)t * a.n_head + kh * gqa + h) * HD + 4u * jg;
    if ((((uintptr_t)a.out | (uintptr_t)a.gate) & 15u) == 0u) {
#pragma unroll
        for (uint32_t T = 0; T < TD; T++) {
            const f4_t g = ldg((const f4_t *)(a.gate + ro + 16u * T));
            f4_t r;
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++) r[i] = acc[T][i] * inv * q4kv_sigmoid(g[i]);
            stg((f4_t *)(a.out + ro + 16u * T), r);
        }
    } else {
#pragma unroll
        for (uint32_t T = 0; T < TD; T++)
#pragma unroll
            for (uint32_t i = 0; i < 4u; i++)
                stg(a.out + ro + 16u * T + i,
                    acc[T][i] * inv * q4kv_sigmoid(ldg(a.gate + ro + 16u * T + i)));
    }
}

/* Merges the S partials of every split column: HD / 4 lanes per column,
 * four dims each, eight splits' rows in flight. An empty partial has l = 0;
 * one with l = NaN (scores that are not finite) takes part, so that a column's
 * result does not depend on how its tile was cut. */
template <int HD> __global__ __launch_bounds__(256) void qsa_dense_merge_k(Args a) {
    constexpr uint32_t LPC = HD / 4, CPW = 256 / LPC;
    const uint32_t c_hi = a.n_tok * a.gqa - a.T1 * COLS, kh = blockIdx.y;
    const uint32_t i = blockIdx.x * CPW + threadIdx.x / LPC, d = 4u * (threadIdx.x % LPC);
    if (i >= c_hi) return;
    const float *pb = a.part + ((size_t)kh * c_hi + i) * a.S * (HD + PHEAD);
    const uint32_t col = a.T1 * COLS + i, t = col / a.gqa, h = col - t * a.gqa;
    const size_t ro = ((size_t)t * a.n_head + kh * a.gqa + h) * HD + d;
    float g[4];
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) g[k] = ldg(a.gate + ro + k);
    float M = -INFINITY, L = 0.f;
    f4_t acc = {0.f, 0.f, 0.f, 0.f};
    for (uint32_t s0 = 0; s0 < a.S; s0 += 8u) {
        f2_t ml[8];
        f4_t v[8];
#pragma unroll
        for (uint32_t k = 0; k < 8u; k++) {
            const float *r = pb + (size_t)min(s0 + k, a.S - 1u) * (HD + PHEAD);
            ml[k] = ldg((const f2_t *)r);
            v[k] = ldg((const f4_t *)(r + PHEAD + d));
        }
        float mn = M;
#pragma unroll
        for (uint32_t k = 0; k < 8u; k++)
            if (s0 + k < a.S && ml[k][1] != 0.f) mn = max2(mn, ml[k][0]);
        const float f = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M - mn);
        L *= f;
        acc *= f;
        M = mn;
#pragma unroll
        for (uint32_t k = 0; k < 8u; k++) {
            if (s0 + k < a.S && ml[k][1] != 0.f) {
                const float w = __builtin_amdgcn_exp2f(ml[k][0] - mn);
                L += w * ml[k][1];
                acc += w * v[k];
            }
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) {
        const float r = L != 0.f ? acc[k] / L : 0.f;
        stg(a.out + ro + k, r * q4kv_sigmoid(g[k]));
    }
}

template <int KIND, int HD> void launch(const Args &a) {
    const uint32_t grid = (a.T1 + (a.n_tiles - a.T1) * a.S) * a.n_kvh;
    const bool prof = q4kv_prof_open();
    qsa_dense_k<KIND, HD><<<grid, NTHR, 0, q4kv_stream>>>(a);
    q4kv_prof_close(prof);
    if (a.T1 < a.n_tiles) {
        const uint32_t cpw = 256u / (HD / 4u), c_hi = a.n_tok * a.gqa - a.T1 * COLS;
        qsa_dense_merge_k<HD><<<dim3((c_hi + cpw - 1u) / cpw, a.n_kvh), 256, 0, q4kv_stream>>>(a);
    }
}

/* Which tiles to split, and into how many pieces. A workgroup fills a CU, so
 * a launch of few tiles leaves CUs idle, and a causal launch of some hundred
 * waits for its longest tile. The cost of a choice, in passes: the longest
 * piece or the CUs' share, rounded up to whole rounds of workgroups where
 * the tiles are alike; a workgroup's start and end (START); the
 * merge launch (MERGE) and the partials, 128 KB written and read per piece
 * (PART). */
constexpr uint32_t N_CU = 256, MAX_SPLIT = 64;
constexpr float START = 4.f, MERGE = 3.f, PART = 0.04f;

void plan(Args &a, uint32_t hd, size_t cap) {
    a.S = 1u;
    a.T1 = a.T2 = a.n_tiles;
    const uint32_t pt = 8192u / hd;
    auto passes = [&](uint32_t tile) {
        const uint64_t cl = std::min<uint64_t>((uint64_t)(tile + 1u) * COLS, (uint64_t)a.n_tok * a.gqa) - 1u;
        const uint64_t n = std::min<uint64_t>(a.kv_base + cl / a.gqa + 1u, a.max_kv);
        return (uint32_t)((n + pt - 1u) / pt);
    };
    const float n_lo = (float)passes(0u), n_hi = (float)passes(a.n_tiles - 1u);
    const float tiles = (float)a.n_tiles * a.n_kvh, total = tiles * 0.5f * (n_lo + n_hi);
    if (!a.part || a.n_kvh > 65535u) return;
    float best = 1e30f;
    const float spread = (n_hi - n_lo) / n_hi;
    static const uint32_t cand[] = {1u, 2u, 3u, 4u, 6u, 8u, 12u, 16u, 24u, 32u, 48u, MAX_SPLIT};
    for (uint32_t S : cand) {
        if (S > 1u && 2u * S > (uint32_t)n_hi) break;
        for (uint32_t k = 0; k < 4u; k++) { /* split the last 4 - k quarters of the tiles */
            const float thr = n_lo + (n_hi - n_lo) * k / 4.f;
            const uint32_t T1 = S == 1u ? a.n_tiles : (uint32_t)((uint64_t)a.n_tiles * k / 4u);
            const float n_split = (float)(a.n_tiles - T1) * a.n_kvh;
            const uint64_t rows = ((uint64_t)a.n_tok * a.gqa - (uint64_t)T1 * COLS) * a.n_kvh * S;
            if (S > 1u && rows * (hd + PHEAD) > cap) continue;
            const float longest = (S == 1u ? n_hi : std::max(n_hi / S, T1 ? thr : 0.f)) + START;
            const float wgs = tiles + n_split * (S - 1u);
            const float even = (total + wgs * START) / N_CU;
            const float rounds = std::ceil(wgs / N_CU) * ((total / wgs) + START);
            float cost = std::max(longest, even + (1.f - spread) * (rounds - even));
            if (S > 1u) cost = 1.03f * cost + MERGE + n_split * S * PART * (hd / 256.f);
            if (cost < best) {
                best = cost;
                a.S = S;
                a.T1 = T1;
            }
            if (S == 1u) break;
        }
    }
    a.T2 = a.T1;
    if (a.S > 1u) {
        while (a.T2 > 0u && passes(a.T2 - 1u) * a.S > (uint32_t)n_hi) {
            /* unsplit tiles longer than a piece go first */
            const uint32_t step = std::max(1u, a.T2 / 64u);
            a.T2 -= std::min(step, a.T2);
        }
    }
    if (a.T1 == a.n_tiles) a.S = 1u;
}

} // namespace

bool q4kv_dense_takes(int kind, uint32_t hd, uint32_t n_tok, uint32_t n_kvh, uint32_t gqa,
                      uint32_t max_n, bool rows16) {
    if (kind != Q4KV_Q8 && kind != Q4KV_F16) return false;
    if (hd != 256u && hd != 128u && hd != 64u) return false;
    if (!rows16 || !max_n) return false;
    const uint64_t cols = (uint64_t)n_tok * gqa;
    if ((cols / COLS + 1u) * n_kvh >= 0x1000000u) return false;
    static const char *force = getenv("Q4KV_DENSE"); /* 0: never, 1: every shape it can */
    if (force) return force[0] != '0';
    /* More heads than the other kernels tile: at any size (the general
     * kernel takes 1.3 to 70 times as long). Otherwise where the other
     * kernels' row slots (KV heads x head groups x attended positions) pass
     * a limit: a launch costs this kernel 7 to 13 us however small.
     * 256 dims, 280 thousand: 24 / 2 heads, 64 tokens: 22.9 against 21.6 us
     * over 300 positions, 29.3 against 34.7 over 1000; 16 / 2 heads, 64
     * tokens: 27.6 against 23.8 over 1000, 37.3 against 46.7 over 4000.
     * 64 and 128 dims (q4kv_rows.hip), 160 thousand: 32 / 8 heads of 128
     * dims: 13.6 against 12.1 us for 8 tokens over 1000 positions, 30.7
     * against 32.1 for 2 over 16000, 32.0 against 86.9 for 8.
     * And where a column tile stands for enough of those slots: a few tokens
     * leave most of its 128 columns empty, and one tile of a long cache is cut
     * into MAX_SPLIT pieces at most. 8 heads per KV head, us by tokens, this
     * kernel against the others: q8_0, 2 KV heads, 130 thousand positions: 2:
     * 165 / 65, 4: 167 / 84, 8: 170 / 149, 16: 173 / 299; 40 thousand: 4: 66 /
     * 48, 8: 69 / 55; 8 KV heads of 4, 40 thousand: 2: 106 / 55, 4: 107 / 93, 6:
     * 108 / 116; f16, 2 KV heads, 130 thousand: 2: 116 / 76, 3: 117 / 99, 6: 119 /
     * 169; q8_0 of 128 dims, 130 thousand: 2: 95 / 64, 4: 96 / 89, 6: 97 / 119. */
    if (gqa > 16u) return true;
    if (n_tok < 2u) return false;
    const uint32_t hg = gqa > 8u ? 2u : 1u;
    const uint64_t slots = (uint64_t)n_tok * n_kvh * hg * (max_n - std::min<uint64_t>(max_n, n_tok) / 2u);
    const float tiles = (float)((cols + COLS - 1u) / COLS) * n_kvh; /* and the CUs that they fill */
    const float per_tile = (float)n_tok * n_kvh * hg / tiles * std::min(1.f, tiles * MAX_SPLIT / N_CU);
    if (slots <= (hd == 256u ? 280000u : 160000u)) return false;
    if (kind == Q4KV_F16 || hd == 64u) return per_tile > 1.5f;
    if (hd == 128u) return per_tile > 2.f;
    /* the others fall back past a size: 6 tokens, 2 KV heads, 130 thousand
     * positions: 163 / 222; 3 tokens, 8 KV heads, 60 thousand: 146 / 173 (40
     * thousand: 105 / 78); 12 heads per KV head, 3 tokens: 40 thousand 66 / 60,
     * 60 thousand 87 / 117 */
    return per_tile > (gqa > 8u ? 3.f : 4.f) || (per_tile > 2.5f && slots > (gqa > 8u ? 600000u : 1300000u));
}

bool q4kv_dense_launch(int kind, uint32_t hd, const float *q, const void *kc, const void *vc,
                       const float *gate, float *out, float *part, size_t cap, uint32_t n_head,
                       uint32_t n_kvh, uint32_t n_tok, uint32_t kv_base, uint32_t max_kv,
                       float scale_log2) {
    Args a = {};
    a.kc = (const uint8_t *)kc;
    a.vc = (const uint8_t *)vc;
    a.q = q;
    a.gate = gate;
    a.out = out;
    a.part = part;
    a.n_head = n_head;
    a.n_kvh = n_kvh;
    a.gqa = n_head / n_kvh;
    a.n_tok = n_tok;
    a.kv_base = kv_base;
    a.max_kv = max_kv;
    a.n_tiles = (uint32_t)(((uint64_t)n_tok * a.gqa + COLS - 1u) / COLS);
    a.scale_log2 = scale_log2;
    plan(a, hd, cap);
    if (kind == Q4KV_Q8)
        hd == 256u ? launch<Q4KV_Q8, 256>(a) : hd == 128u ? launch<Q4KV_Q8, 128>(a) : launch<Q4KV_Q8, 64>(a);
    else
        hd == 256u ? launch<Q4KV_F16, 256>(a) : hd == 128u ? launch<Q4KV_F16, 128>(a) : launch<Q4KV_F16, 64>(a);
    return q4kv_launch_ok("qsa dense prefill");
}

/* n_items counts, then (m, l) pairs from an even offset (they are read and
 * written as 8 bytes) */
static size_t band_ml_at(uint32_t n_items) { return ((size_t)n_items + 1u) / 2u * 2u; }
size_t q4kv_band_floats(uint32_t n_items, uint32_t gqa) {
    return band_ml_at(n_items) + (size_t)n_items * 2u * gqa;
}

bool q4kv_band_launch(AttnArgs &a, uint32_t n_items, float *part) {
    const uint32_t gqa = a.n_head / a.n_kvh;
    Args b = {};
    b.kc = a.kc;
    b.vc = a.vc;
    b.q = a.q;
    b.out = a.out;
    b.n_head = a.n_head;
    b.n_kvh = a.n_kvh;
    b.gqa = gqa;
    b.n_tok = n_items / a.n_kvh;
    b.max_kv = a.max_kv;
    b.toks = std::min(COLS / gqa, BAND_TOKS);
    b.n_tiles = b.T1 = b.T2 = (b.n_tok + b.toks - 1u) / b.toks;
    b.S = 1u;
    b.scale_log2 = a.scale_log2;
    b.idx = a.idx;
    b.tok_stride = a.tok_stride;
    b.kvh_stride = a.kvh_stride;
    b.width = a.width;
    b.band_nb = a.band_nb = (int32_t *)part;
    b.band_ml = a.band_ml = part + band_ml_at(n_items);
    qsa_dense_k<Q4KV_Q8, 256, true><<<b.n_tiles * a.n_kvh, NTHR, 0, q4kv_stream>>>(b);
    return q4kv_launch_ok("qsa band");
}
