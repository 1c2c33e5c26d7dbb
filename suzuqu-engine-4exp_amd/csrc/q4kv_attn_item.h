/*
 * q4kv_attn_item.h -- what the attention kernels' translation units share:
 * launch arguments, work items (one token or sequence and KV head, from the
 * direct arguments or a descriptor) and small lane arithmetic.
 */
#ifndef Q4KV_ATTN_ITEM_H
#define Q4KV_ATTN_ITEM_H
#include <hip/hip_runtime.h>
#include <math.h>
#include <stddef.h>

#include "q4kv_internal.h"

extern "C" {
#include "q4kv.h"
}

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));

/* MODE_STEP: MODE_BATCH over q4kv_step_desc entries, with the token's K/V
 * append done by the same launch (fast q8_0 kernel only). */
/* MODE_PSTEP: MODE_STEP over q4kv_prep_step_desc entries, with the query
 * and key preparation (RMSNorm + RoPE) done in the kernel. */
enum { MODE_DENSE = 0, MODE_INDEXED = 1, MODE_BATCH = 2, MODE_STEP = 3, MODE_PSTEP = 4 };
#define IS_STEP(M) ((M) == MODE_STEP || (M) == MODE_PSTEP)
#define IS_BATCH(M) ((M) == MODE_BATCH || IS_STEP(M))

struct AttnArgs {
    const uint8_t *kc, *vc;
    const float *q, *gate;
    float *out;
    const int32_t *idx;
    uint64_t tok_stride, kvh_stride;
    const q4kv_seq_desc *seqs;
    uint32_t desc_stride; /* bytes between descriptors (64, or 96 for steps) */
    float *part;
    uint32_t width, kv_base, max_kv;
    uint32_t n_head, n_kvh, hd;
    uint32_t S, cps, item0;
    float scale_log2;
    /* MODE_PSTEP */
    uint32_t n_rot;
    float rope_base, eps;
    /* prefill band (MODE_INDEXED): per item, the list entries before its
     * band (the slab kernel's list length) and the band's (m, l) per head;
     * the band's unnormalised output rows are in out */
    int32_t *band_nb;
    float *band_ml;
    /* XCD grouping (xcd_slot; 1D grid when xgrp > 0): xgrp (token, split)
     * groups, each run by its n_kvh KV heads' workgroups on one XCD */
    uint32_t xgrp;
    /* the held append of one token's K/V rows ([n_kvh][hd] fp32 each) at
     * the device position *app_pos (qsa_q8d256_k with APP) */
    const float *app_k, *app_v;
    const int32_t *app_pos;
};

struct Item {
    const uint8_t *kc, *vc;
    const float *q, *gate;
    float *out;
    const int32_t *list;
    uint32_t n, max_kv;
    /* index-load source and mask: (list, ~0) for a list, (any readable word,
     * 0) for a dense item, so that loads and selects need no branch */
    const int32_t *lsrc;
    uint32_t lmask;
    /* MODE_STEP: this KV head's new K/V rows and their position */
    const float *knew, *vnew;
    uint32_t pos_new;
    /* MODE_PSTEP: RMSNorm weights; q rows are [q | gate] (head stride 2*hd) */
    const float *wnq, *wnk;
};

template <int MODE>
__device__ static inline Item resolve_item(const AttnArgs &a, uint32_t item) {
    const uint32_t kh = item % a.n_kvh, t = item / a.n_kvh;
    const uint32_t gqa = a.n_head / a.n_kvh;
    const size_t hoff = (size_t)kh * gqa * a.hd;
    Item it;
    it.knew = it.vnew = nullptr;
    it.wnq = it.wnk = nullptr;
    it.pos_new = ~0u;
    if (IS_BATCH(MODE)) {
        /* every descriptor word this mode reads, in one batch of scalar loads
         * issued together (field-by-field loads behind the pointer tests
         * cost extra dependent round trips before the first index load) */
        constexpr uint32_t NW = MODE == MODE_PSTEP ? 28u : IS_STEP(MODE) ? 21u : 15u;
        const uint32_t *dw =
            (const uint32_t *)((const uint8_t *)a.seqs + (size_t)t * a.desc_stride);
        uint32_t w[NW];
#pragma unroll
        for (uint32_t i = 0; i < NW; i++) w[i] = ldg(dw + i);
        /* consume every word here so none of the loads sinks to its use */
#pragma unroll
        for (uint32_t i = 0; i < NW; i++) asm volatile("" ::"s"(w[i]));
        auto word = [&](uint32_t byte_off) {
            return (uintptr_t)w[byte_off / 4u] | ((uintptr_t)w[byte_off / 4u + 1u] << 32);
        };
        /* descriptor pointers as global-address-space pointers: accesses
         * through them need no flat instructions */
        static_assert(offsetof(q4kv_seq_desc, kcache) == 0 && offsetof(q4kv_seq_desc, vcache) == 8 &&
                          offsetof(q4kv_seq_desc, q) == 16 && offsetof(q4kv_seq_desc, gate) == 24 &&
                          offsetof(q4kv_seq_desc, out) == 32 && offsetof(q4kv_seq_desc, idx) == 40 &&
                          offsetof(q4kv_seq_desc, n_sel) == 48 &&
                          offsetof(q4kv_seq_desc, idx_kvh_stride) == 52 &&
                          offsetof(q4kv_seq_desc, max_kv) == 56,
                      "q4kv_seq_desc layout");
        static_assert(offsetof(q4kv_step_desc, k) == 64 && offsetof(q4kv_step_desc, v) == 72 &&
                          offsetof(q4kv_step_desc, pos) == 80,
                      "q4kv_step_desc layout");
        static_assert(offsetof(q4kv_prep_step_desc, wn_q) == 96 &&
                          offsetof(q4kv_prep_step_desc, wn_k) == 104,
                      "q4kv_prep_step_desc layout");
        const float *gate = q4kv_gptr<const float>(word(24));
        const int32_t *idx = q4kv_gptr<const int32_t>(word(40));
        const uint32_t n_sel = w[12];
        it.kc = q4kv_gptr<const uint8_t>(word(0));
        it.vc = q4kv_gptr<const uint8_t>(word(8));
        it.q = q4kv_gptr<const float>(word(16)) + hoff * (MODE == MODE_PSTEP ? 2u : 1u);
        it.gate = gate ? gate + hoff : nullptr;
        it.out = q4kv_gptr<float>(word(32)) + hoff;
        it.max_kv = w[14];
        it.list = idx ? idx + (size_t)kh * w[13] : nullptr;
        it.n = idx ? n_sel : (n_sel < it.max_kv ? n_sel : it.max_kv);
        it.lsrc = idx ? it.list : (const int32_t *)a.seqs;
        it.lmask = idx ? ~0u : 0u;
        if (IS_STEP(MODE)) {
            it.knew = q4kv_gptr<const float>(word(64)) + (size_t)kh * a.hd;
            it.vnew = q4kv_gptr<const float>(word(72)) + (size_t)kh * a.hd;
            it.pos_new = w[20];
        }
        if (MODE == MODE_PSTEP) {
            it.wnq = q4kv_gptr<const float>(word(96));
            it.wnk = q4kv_gptr<const float>(word(104));
        }
    } else {
        const size_t qo = (size_t)t * a.n_head * a.hd + hoff;
        it.kc = a.kc;
        it.vc = a.vc;
        it.q = a.q + qo;
        it.gate = a.gate ? a.gate + qo : nullptr;
        it.out = a.out + qo;
        it.max_kv = a.max_kv;
        if (MODE == MODE_INDEXED) {
            it.list = a.idx + t * a.tok_stride + kh * a.kvh_stride;
            it.n = a.width;
            it.lsrc = it.list;
            it.lmask = ~0u;
        } else {
            const uint32_t nkv = a.kv_base + t + 1u;
            it.list = nullptr;
            it.n = nkv < a.max_kv ? nkv : a.max_kv;
            it.lsrc = nullptr;
            it.lmask = 0u;
        }
    }
    return it;
}

/* v + (value of the lane 32 apart): the swap leaves each lane's own value in
 * one result and its partner's in the other, so their sum needs no select. */
__device__ static inline float pair32_sum(float v) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                              false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
/* max(a, b) for non-NaN operands in one v_med3_f32 (fmaxf adds NaN-quieting
 * canonicalisations of both operands). */
__device__ static inline float fmax2(float a, float b) {
    return __builtin_amdgcn_fmed3f(a, b, INFINITY);
}

/* Reductions across the four 16-lane rows (v_permlane16_swap: the lane 16
 * apart within each half; v_permlane32_swap: the lane 32 apart). */
__device__ static inline float sum16(float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ static inline float max16(float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmax2(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ static inline float max32(float v) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmax2(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
/* v + (value of lane c + 8 mod 16 in the same DPP row): hi + lo columns */
__device__ static inline float add_ror8(float v) {
    return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xF, 0xF, true));
}
/* fp16 halves of a packed word as fp32 (folded into v_fma_mix operands) */
__device__ static inline float h2lo(uint32_t w) { return (float)__builtin_bit_cast(h2_t, w)[0]; }
__device__ static inline float h2hi(uint32_t w) { return (float)__builtin_bit_cast(h2_t, w)[1]; }
/* x, y -> two fp16 by truncation, packed (v_cvt_pkrtz_f16_f32) */
__device__ static inline uint32_t pkrtz(float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x, y));
}
/* fp16 hi part of (x, y) (nsel = 0) or the fp16 residual x - hi (nsel = -1),
 * packed; hi by truncation, so hi + lo carries ~21 bits. */
__device__ static inline uint32_t split_pk(float x, float y, float nsel) {
    const uint32_t h = pkrtz(x, y);
    return pkrtz(__builtin_fmaf(nsel, h2lo(h), x), __builtin_fmaf(nsel, h2hi(h), y));
}

/* The timing of attention launches, while q4kv_prof_begin has armed it: events
 * around the attention kernel (and the window's, not the merges). */
bool q4kv_prof_open(void);
void q4kv_prof_close(bool open);

/* q8_0 V as the matrix products take it: v x scale in two fp16 parts, exact
 * for every scale below 512 (an int8 times an fp16: 19 bits, none below 2^-24;
 * 128 x 511.75 is still fp16). Whoever meets a larger finite scale goes over to
 * v x scale / 128 from those rows on, its accumulators with it (exact down to
 * 2^-18, 2^-34 of the V that asks for it), and multiplies back at the end. At
 * a fixed 1 / 128, small V lose bits: 1.5e-3 of the result at V x 1e-3, where
 * this leaves 3e-7 as at any size. The look at every pass's scales costs 1 %
 * (one-token decode, listed prefill) or less (dense prefill), in the branch of
 * the running maximum where there is room; starting over with / 128 after a
 * loop that ended in inf - inf cost more (registers). */
struct VScale {
    uint32_t m = 0x3C003C00u, c = 0xE480E480u; /* 1, -1152; 1 / 128, -9 */
    __device__ bool big() const { return m != 0x3C003C00u; }
    __device__ void divide() {
        m = 0x20002000u;
        c = 0xC880C880u;
    }
    /* v (/ 128), exact, of x = 1024 + biased byte */
    __device__ h2_t value(h2_t x) const {
        return __builtin_elementwise_fma(x, __builtin_bit_cast(h2_t, m), __builtin_bit_cast(h2_t, c));
    }
    __device__ float undo() const { return big() ? 128.f : 1.f; }
};
constexpr float VSCALE_STEP = 0.0078125f;
/* a finite fp16 of magnitude 512 or more */
__device__ static inline bool q4kv_big_scale(uint32_t s) { return (s & 0x7C00u) - 0x6000u < 0x1C00u; }

/* Decode attention at 64 and 128 head dims (q4kv_rows.hip): whether it takes
 * a shape, and its launches (mode: MODE_DENSE, MODE_INDEXED or MODE_BATCH).
 * It uses at most Q4KV_ROWS_PART floats of partials. */
#define Q4KV_ROWS_PART ((size_t)4 << 20)
bool q4kv_rows_takes(int kind, uint32_t hd, uint32_t gqa, bool rows16);
bool q4kv_rows_launch(int kind, int mode, const AttnArgs &a, uint32_t n_items, uint32_t max_n,
                      float *part, size_t cap);

/* Listed attention of many items over a q8_0 cache, hd 256, up to 16 query
 * heads per KV head (q4kv_sparse.hip): a.S splits of each list, partials in
 * natural column order; a.xgrp: the tokens, where a token's KV heads share its
 * list and go to one XCD, or 0. */
bool q4kv_sparse_launch(const AttnArgs &a, uint32_t n_items);

/* The shared recent window of consecutive prefill tokens' lists (q8_0, hd
 * 256; q4kv_dense.hip): each token's band of consecutive positions at its
 * list's end is attended as dense tiles. Sets a.band_nb (list entries before
 * the band) and a.band_ml ((m, l) per head), in part, and leaves the bands'
 * unnormalised rows in a.out. */
size_t q4kv_band_floats(uint32_t n_items, uint32_t gqa);
bool q4kv_band_launch(AttnArgs &a, uint32_t n_items, float *part);

#endif
