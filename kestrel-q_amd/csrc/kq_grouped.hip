/*
 * kq_grouped.hip — the multi-token (prefill) MoE layer as grouped expert
 * GEMMs on MFMA: a stable token->expert permutation, one gate/up + SwiGLU
 * pass and one down pass per expert over all of its tokens, and the ordered
 * combine with the sigmoid-gated shared expert.
 *
 * The reference runs the layer token by token (kq_moe_execute_common,
 * src/kq_moe_qwen38.c:666-865): for each token, route, then for every
 * selected expert in ascending id g = Wg x, u = Wu x, a = swiglu(g, u),
 * o = Wd a, routed_sum += o * w (:722-765), and out = routed_sum +
 * sigmoid(wsg . x) * shared(x) (:771-828). With T tokens every expert's
 * weights would stream once per token that selects it. Here each expert's
 * weights stream once for all of its tokens:
 *
 *   permute  offsets[e], and the (token, slot) pairs of expert e at
 *            positions offsets[e].. in ascending token order (a stable
 *            counting sort; bit-exact by construction)
 *   gate/up  act[pos] = swiglu(Wg_e x_t, Wu_e x_t) for every position of e
 *   down     o[pos] = Wd_e act[pos]
 *   combine  out[t] = sum over t's slots in ascending expert id of
 *            o[pos] * w, then + sigmoid(shared logit) * o_shared[t]
 *
 * GEMM numerics. Weight codes are small integers, exact in fp16, so the
 * quantized weights enter the MFMA exactly:
 *   Q4_K  the 6-bit sub-block scale s is folded into the code (s * q <=
 *         945, exact) with one packed fp16 FMA that also removes the
 *         1024 exponent bias of the byte->fp16 conversion; the super-block
 *         scale d multiplies the fp32 accumulator once per 256 columns and
 *         the dmin * m term is a second small MFMA against per-sub-block
 *         activation sums;
 *   Q6_K  the code q - 32 is exact; each 16-column sub-block is one
 *         16x16x16 MFMA step whose fp32 result is scaled by d * sc.
 * Activations are split per token into fp16 hi + lo (x = hi + lo to ~22
 * bits) after an exact power-of-two scaling that puts the row's largest
 * magnitude in [2^14, 2^15), so neither part overflows and small rows keep
 * their precision; every MFMA accumulates in fp32. Outputs are compared
 * with the CPU by tolerance (per element, 1e-4 absolute or 1e-3 relative).
 *
 * MFMA operands: A = activations (16 tokens x K), B = weights (K x 16
 * rows); lane l holds token / row l % 16 and a k-group l / 16, and the
 * result D[token][row] leaves lane l with row l % 16 of tokens
 * 4 (l / 16) .. + 3. Which hidden columns a k-slot of a step holds is free
 * as long as A and B agree; it is chosen per format so that each lane's
 * weight bytes are contiguous and share one scale.
 */
#include "kq_launch.h"
#include "kq_stage.h"
#include "kq_device.h"
#include "kq_dma.h"
#include "kq_mfma.h"

namespace {

using namespace kq::mf;

constexpr uint32_t kTile = 16;          /* tokens per M-chunk, rows per N-tile */

__device__ __forceinline__ uint32_t as_u(h2 v) { return __builtin_bit_cast(uint32_t, v); }

__device__ __forceinline__ float wave_max_abs(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, KQ_WAVE));
    return v;
}

/* ------------------------------------------------------------------ */
/* formats */

template <uint32_t FMT>
struct Fmt;

/* Q4_K: 144 B per 256 columns (d, dmin, 12 B of 6-bit scales/mins, 128 B
 * of nibbles; src/kq_numeric.c:223-277). Lane k-group g reads nibble group
 * g (qs bytes 32g..32g+31: sub-blocks 2g in the low nibbles, 2g+1 in the
 * high) of its row; step s (0..7) of a block covers hidden columns
 * 64g + 8s .. +7, low nibbles for s < 4, high nibbles for s >= 4. */
template <>
struct Fmt<KQ_LAUNCH_Q4_K> {
    static constexpr uint32_t kUnit = 256u;       /* columns per pass iteration */
    static constexpr uint32_t kUnitBytes = 144u;
    static constexpr bool kSums = true;           /* 32-column activation sums */
    static constexpr bool kK32 = true; /* 16x16x32 steps, b128 activation reads */
    struct Raw {
        uint4 hd, qa, qb;
    };
    __device__ static __forceinline__ Raw load(KqBuf w, uint32_t boff, uint32_t g) {
        Raw r;
        r.hd = kq_ld128(w, boff, 0u);
        r.qa = kq_ld128(w, boff + 16u + 32u * g, 0u);
        r.qb = kq_ld128(w, boff + 32u + 32u * g, 0u);
        return r;
    }
};

/* Q6_K: 210 B per 256 columns (ql[128], qh[64], int8 sc[16], f16 d; GGML
 * layout). Sub-block s = 8n + 2q + h (half n, quarter q, 16-column half
 * h) is one 16x16x16 step; lane k-group g holds its columns 4g .. 4g+3,
 * i.e. hidden 128n + 32q + 16h + 4g .. +3, whose codes come from the ql
 * dwords at 64n + 16h + 4g (q = 0, 2) and 64n + 32 + 16h + 4g (q = 1, 3)
 * and the qh dword at 128 + 32n + 16h + 4g. A block at an offset of 2 mod
 * 4 is read through aligned windows re-aligned with a byte funnel shift;
 * no window leaves the block. */
template <>
struct Fmt<KQ_LAUNCH_Q6_K> {
    static constexpr uint32_t kBytes = 210u;
    static constexpr uint32_t kUnit = 256u;
    static constexpr uint32_t kUnitBytes = 210u;
    static constexpr bool kSums = false;
    static constexpr bool kK32 = false;
    struct Raw {
        kq_u32x2 w[4][3]; /* [n * 2 + h][ql A, ql B, qh] */
        uint4 sc;         /* window over sc[16] */
        uint32_t sc_tail, d, sh;
    };
    __device__ static __forceinline__ Raw load(KqBuf w, uint32_t boff, uint32_t g) {
        Raw r;
        r.sh = boff & 3u;
        const uint32_t base = boff - r.sh;
#pragma unroll
        for (uint32_t nh = 0; nh < 4u; ++nh) {
            const uint32_t n = nh >> 1, h = nh & 1u;
            const uint32_t oa = 64u * n + 16u * h + 4u * g;
            r.w[nh][0] = kq_ld64(w, base + oa, 0u);
            r.w[nh][1] = kq_ld64(w, base + oa + 32u, 0u);
            r.w[nh][2] = kq_ld64(w, base + 128u + 32u * n + 16u * h + 4u * g, 0u);
        }
        /* sc[16] at 192: [192, 208) when aligned, else [190, 210); the
         * tail word is loaded on every path (a branch here would split the
         * wave) and only used for an unaligned block */
        r.sc = kq_ld128(w, base + 192u, 0u);
        r.sc_tail = kq_ld32(w, base + 208u, 0u);
        r.d = kq_ld16(w, boff + 208u, 0u);
        return r;
    }
};

/* Q8_0: 34 B per 32 columns (f16 d, 32 int8 codes; src/kq_numeric.c:
 * 176-196). An iteration takes two blocks (64 columns); each block is one
 * 16x16x32 step, lane k-group g holding its columns 8g .. 8g + 7, i.e. code
 * bytes 2 + 8g .. 9 + 8g. The first block's codes start at 2 mod 4, so they
 * come from a 12-byte window re-aligned by two bytes; each scale is half of
 * an aligned dword. Rows are whole units of 68 B, so a unit starts 4-byte
 * aligned. */
template <>
struct Fmt<KQ_LAUNCH_Q8_0> {
    static constexpr uint32_t kUnit = 64u;
    static constexpr uint32_t kUnitBytes = 68u;
    static constexpr bool kSums = false;
    static constexpr bool kK32 = true;
    struct Raw {
        kq_u32x3 c[2]; /* code windows of the two blocks */
        uint32_t d[2]; /* dwords holding the scales */
    };
    __device__ static __forceinline__ Raw load(KqBuf w, uint32_t uoff, uint32_t g) {
        Raw r;
#pragma unroll
        for (uint32_t bb = 0; bb < 2u; ++bb) {
            const uint32_t a = uoff + 34u * bb + 2u + 8u * g; /* codes */
            r.c[bb] = kq_ld96(w, a & ~3u, 0u);
            r.d[bb] = kq_ld32(w, (uoff + 34u * bb) & ~3u, 0u);
        }
        return r;
    }
};

/* Q5_1: 24 B per 32 columns (f16 d, f16 m, 32 high bits qh, 16 bytes of
 * nibbles: low nibble of byte i = element i, high = element i + 16, bit i
 * of qh = bit 4 of element i; src/kq_numeric.c:197-222). Four blocks per
 * iteration (96 B); lane k-group g holds elements 8g .. 8g + 7: nibbles of
 * bytes 8(g & 1) .. +7 (low for g < 2, high otherwise) and qh byte g. */
template <>
struct Fmt<KQ_LAUNCH_Q5_1> {
    static constexpr uint32_t kUnit = 128u;
    static constexpr uint32_t kUnitBytes = 96u;
    static constexpr bool kSums = true;
    static constexpr bool kK32 = true;
    struct Raw {
        kq_u32x2 q[4];
        uint32_t dm[4], qh[4];
    };
    __device__ static __forceinline__ Raw load(KqBuf w, uint32_t uoff, uint32_t g) {
        Raw r;
#pragma unroll
        for (uint32_t bb = 0; bb < 4u; ++bb) {
            const uint32_t o = uoff + 24u * bb;
            r.dm[bb] = kq_ld32(w, o, 0u);
            r.qh[bb] = kq_ld32(w, o + 4u, 0u);
            r.q[bb] = kq_ld64(w, o + 8u + 8u * (g & 1u), 0u);
        }
        return r;
    }
};

/* ------------------------------------------------------------------ */
/* LDS image of one M-chunk of activations */

template <uint32_t FMT, uint32_t KDIM>
struct Stage {
    /* row pitch in fp16: b128 reads (K32 steps) want a 16-byte skew per
     * row, b64 reads an 8-byte one, so that 8 / 16 lanes on consecutive
     * rows hit distinct banks */
    static constexpr uint32_t kPitch = KDIM + (Fmt<FMT>::kK32 ? 8u : 4u);
    static constexpr uint32_t kSub = KDIM / 32u; /* Q4_K sub-blocks per row */
    static constexpr uint32_t kSxPitch = kSub + 8u;
    static constexpr bool kSums = Fmt<FMT>::kSums;
    __align__(16) _Float16 xh[kTile * kPitch];
    __align__(16) _Float16 xl[kTile * kPitch];
    __align__(16) _Float16 sxh[kSums ? kTile * kSxPitch : 4];
    __align__(16) _Float16 sxl[kSums ? kTile * kSxPitch : 4];
    int sig[kTile];
};

/* Stage columns col0 .. col0 + KSL - 1 of rows src_row[i] (or zeros where
 * negative) of X [*, KDIM]: scale by 2^sig (the row's largest magnitude,
 * over all KDIM columns, into [2^14, 2^15), so every slice of a row gets
 * the same scale), split into fp16 hi + lo and, for formats with a min
 * term, form the 32-column sums of the scaled row times 2^-5 (so they fit
 * fp16), also split. One wave per row; lane l holds the float4 column
 * groups l, l + 64, ..., so that both the global reads and the LDS writes
 * of a wave are contiguous (no bank conflicts). Returns true if a
 * non-finite input was seen. col0 and KSL are multiples of 32. */
template <uint32_t FMT, uint32_t KDIM, uint32_t KSL>
__device__ bool stage_slice(Stage<FMT, KSL> &st, const float *__restrict__ X, uint32_t col0,
                            const int *src_row, uint32_t wave, uint32_t nwaves, uint32_t lane) {
    using S = Stage<FMT, KSL>;
    constexpr uint32_t NQ = (KDIM + 255u) / 256u;   /* float4 groups per lane, whole row */
    constexpr uint32_t NQS = (KSL + 255u) / 256u + (KSL % 256u != 0u ? 1u : 0u); /* a slice */
    bool bad = false;
    for (uint32_t i = wave; i < kTile; i += nwaves) {
        const int src = src_row[i];
        const float4 *p = (const float4 *)(X + (size_t)(src < 0 ? 0 : src) * KDIM) + lane;
        int sig;
        bool any_nf = false;
        if (col0 == 0u) {
            /* the scale, from the whole row (later slices of this chunk reuse
             * it, so every slice gets the same one) */
            float m = 0.0f;
            bool nf = false;
#pragma unroll 8
            for (uint32_t q = 0; q < NQ; ++q) {
                const bool in = src >= 0 && 256u * q + 4u * lane < KDIM;
                const float4 v = in ? p[64u * q] : make_float4(0.f, 0.f, 0.f, 0.f);
                nf |= !kq_isfinite(v.x) || !kq_isfinite(v.y) || !kq_isfinite(v.z) ||
                      !kq_isfinite(v.w);
                m = fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
            }
            bad |= nf;
            m = wave_max_abs(m);
            any_nf = __ballot(nf) != 0ull;
            /* m = f * 2^e, f in [0.5, 1): m * 2^(15 - e) lies in [2^14, 2^15) */
            sig = 0;
            if (!any_nf && m > 0.0f) sig = 15 - __builtin_amdgcn_frexp_expf(m);
            if (any_nf) sig = 0x7fffffff; /* a row staged as zeros */
        } else {
            sig = st.sig[i];
            any_nf = sig == 0x7fffffff;
        }
        const uint32_t q0 = col0 / 256u;
        float4 v[NQS];
#pragma unroll
        for (uint32_t qq = 0; qq < NQS; ++qq) {
            const uint32_t col = 256u * (q0 + qq) + 4u * lane;
            const bool in = src >= 0 && col < KDIM;
            v[qq] = in ? p[64u * (q0 + qq)] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (uint32_t qq = 0; qq < NQS; ++qq) {
            const uint32_t col = 256u * (q0 + qq) + 4u * lane;
            const bool mine = col >= col0 && col < col0 + KSL;
            const float a[4] = {v[qq].x, v[qq].y, v[qq].z, v[qq].w};
            _Float16 hi[4], lo[4];
            float part = 0.0f;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float xs = any_nf ? 0.0f : ldexpf(a[c], sig);
                hi[c] = (_Float16)xs;
                lo[c] = (_Float16)(xs - (float)hi[c]);
                part += xs;
            }
            if (mine) {
                *(h4 *)(st.xh + i * S::kPitch + (col - col0)) = h4{hi[0], hi[1], hi[2], hi[3]};
                *(h4 *)(st.xl + i * S::kPitch + (col - col0)) = h4{lo[0], lo[1], lo[2], lo[3]};
            }
            if constexpr (S::kSums) {
                /* 32-column sums: 8 consecutive lanes hold one */
                part += __shfl_xor(part, 1, KQ_WAVE);
                part += __shfl_xor(part, 2, KQ_WAVE);
                part += __shfl_xor(part, 4, KQ_WAVE);
                if (mine && (lane & 7u) == 0u) {
                    const float s = part * 0.03125f;
                    const _Float16 sh = (_Float16)s;
                    const _Float16 sl = (_Float16)(s - (float)sh);
                    const uint32_t jsb = (col - col0) / 32u;
                    st.sxh[i * S::kSxPitch + jsb] = sh;
                    st.sxl[i * S::kSxPitch + jsb] = sl;
                }
            }
        }
        if (lane == 0u) st.sig[i] = sig;
    }
    return bad;
}

template <uint32_t FMT, uint32_t KDIM>
__device__ bool stage_rows(Stage<FMT, KDIM> &st, const float *__restrict__ X,
                           const int *src_row, uint32_t wave, uint32_t nwaves, uint32_t lane) {
    return stage_slice<FMT, KDIM, KDIM>(st, X, 0u, src_row, wave, nwaves, lane);
}

/* ------------------------------------------------------------------ */
/* one 16-row N-tile of NMAT matrices (gate and up share the activation
 * fragments of every step) against the staged 16-token chunk; acc[m] gets
 * block b of matrix m */

template <uint32_t FMT, uint32_t KDIM, int NMAT>
struct Tile;

template <uint32_t KDIM, int NMAT>
struct Tile<KQ_LAUNCH_Q4_K, KDIM, NMAT> {
    using F = Fmt<KQ_LAUNCH_Q4_K>;
    using S = Stage<KQ_LAUNCH_Q4_K, KDIM>;
    using Raw = F::Raw;

    __device__ static __forceinline__ void block(const Raw (&r)[NMAT], const S &st, uint32_t b,
                                                 uint32_t i, uint32_t g, f4 (&acc)[NMAT],
                                                 bool &malformed) {
        float d[NMAT], dm[NMAT];
        h2 S0[NMAT], C0[NMAT], S1[NMAT], C1[NMAT];
        h4 bm[NMAT];
#pragma unroll
        for (int m = 0; m < NMAT; ++m) {
            d[m] = half_bits(r[m].hd.x);
            const float dmin = half_bits(r[m].hd.x >> 16);
            malformed |= !kq_isfinite(d[m]) || !kq_isfinite(dmin);
            dm[m] = dmin * 32.0f; /* the activation sums carry 2^-5 */
            /* scales of sub-blocks 2g and 2g+1 (src/kq_numeric.c:161-174) */
            const uint32_t u = r[m].hd.y >> (16u * (g & 1u)); /* q[2(g&1)], q[2(g&1)+1] */
            const uint32_t w = r[m].hd.w >> (16u * (g & 1u)); /* q[8+2(g&1)], q[9+2(g&1)] */
            uint32_t s0, s1;
            if (g < 2u) {
                s0 = u & 63u;
                s1 = (u >> 8) & 63u;
            } else {
                s0 = (w & 15u) | ((u >> 2) & 0x30u);
                s1 = ((w >> 8) & 15u) | ((u >> 10) & 0x30u);
            }
            const _Float16 fs0 = (_Float16)(float)s0, fs1 = (_Float16)(float)s1;
            S0[m] = h2{fs0, fs0};
            C0[m] = S0[m] * h2{(_Float16)-1024.0f, (_Float16)-1024.0f};
            S1[m] = h2{fs1, fs1} * h2{(_Float16)0.0625f, (_Float16)0.0625f};
            C1[m] = h2{fs1, fs1} * h2{(_Float16)-64.0f, (_Float16)-64.0f};
            /* mins m_4g .. m_4g+3 for g < 2 (the min-term weights); 0 for g >= 2 */
            const uint32_t mq =
                g == 0u ? (r[m].hd.z & 0x3f3f3f3fu)
                        : (((r[m].hd.w >> 4) & 0x0f0f0f0fu) | ((r[m].hd.z >> 2) & 0x30303030u));
            const h2 one = h2{(_Float16)1.0f, (_Float16)1.0f};
            const h2 neg = h2{(_Float16)-1024.0f, (_Float16)-1024.0f};
            h2 mlo = fma2(bytes_lo(mq), one, neg), mhi = fma2(bytes_hi(mq), one, neg);
            if (g >= 2u) {
                mlo = h2{(_Float16)0.0f, (_Float16)0.0f};
                mhi = mlo;
            }
            bm[m] = h4{mlo.x, mlo.y, mhi.x, mhi.y};
        }
        f4 q[NMAT];
#pragma unroll
        for (int m = 0; m < NMAT; ++m) q[m] = f4{0.f, 0.f, 0.f, 0.f};
        const _Float16 *xh = st.xh + i * S::kPitch + 256u * b + 64u * g;
        const _Float16 *xl = st.xl + i * S::kPitch + 256u * b + 64u * g;
#pragma unroll
        for (uint32_t s = 0; s < 8u; ++s) {
            const h8 ah = *(const h8 *)(xh + 8u * s);
            const h8 al = *(const h8 *)(xl + 8u * s);
#pragma unroll
            for (int m = 0; m < NMAT; ++m) {
                const uint4 &qd = (s & 2u) ? r[m].qb : r[m].qa;
                const uint32_t raw0 = (s & 1u) ? qd.z : qd.x, raw1 = (s & 1u) ? qd.w : qd.y;
                const uint32_t m0 = s < 4u ? kq_and_0f(raw0) : kq_and_f0(raw0);
                const uint32_t m1 = s < 4u ? kq_and_0f(raw1) : kq_and_f0(raw1);
                const h2 Sc = s < 4u ? S0[m] : S1[m], Cc = s < 4u ? C0[m] : C1[m];
                const h2 w0 = fma2(bytes_lo(m0), Sc, Cc), w1 = fma2(bytes_hi(m0), Sc, Cc);
                const h2 w2 = fma2(bytes_lo(m1), Sc, Cc), w3 = fma2(bytes_hi(m1), Sc, Cc);
                const h8 bw = h8{w0.x, w0.y, w1.x, w1.y, w2.x, w2.y, w3.x, w3.y};
                q[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bw, q[m], 0, 0, 0);
                q[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bw, q[m], 0, 0, 0);
            }
            /* keep each step's fragments short-lived: without this the
             * scheduler hoists every step's LDS reads and runs out of VGPRs */
            __builtin_amdgcn_sched_barrier(0);
        }
        /* min term: sum_j m_j * (32-column sums * 2^-5) */
        const uint32_t so = i * S::kSxPitch + 8u * b + 4u * (g & 1u);
        const h4 sh4 = *(const h4 *)(st.sxh + so);
        const h4 sl4 = *(const h4 *)(st.sxl + so);
#pragma unroll
        for (int m = 0; m < NMAT; ++m) {
            f4 mm = {0.f, 0.f, 0.f, 0.f};
            mm = __builtin_amdgcn_mfma_f32_16x16x16f16(sh4, bm[m], mm, 0, 0, 0);
            mm = __builtin_amdgcn_mfma_f32_16x16x16f16(sl4, bm[m], mm, 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[m][t] = fmaf(d[m], q[m][t], fmaf(-dm[m], mm[t], acc[m][t]));
        }
    }
};

template <uint32_t KDIM, int NMAT>
struct Tile<KQ_LAUNCH_Q6_K, KDIM, NMAT> {
    using F = Fmt<KQ_LAUNCH_Q6_K>;
    using S = Stage<KQ_LAUNCH_Q6_K, KDIM>;
    using Raw = F::Raw;

    __device__ static __forceinline__ void block(const Raw (&r)[NMAT], const S &st, uint32_t b,
                                                 uint32_t i, uint32_t g, f4 (&acc)[NMAT],
                                                 bool &malformed) {
        float d[NMAT];
        uint32_t sc[NMAT][4];
#pragma unroll
        for (int m = 0; m < NMAT; ++m) {
            d[m] = half_bits(r[m].d);
            malformed |= !kq_isfinite(d[m]);
            const uint32_t sh = r[m].sh ? 2u : 0u;
            sc[m][0] = kq_align2(r[m].sc.y, r[m].sc.x, sh);
            sc[m][1] = kq_align2(r[m].sc.z, r[m].sc.y, sh);
            sc[m][2] = kq_align2(r[m].sc.w, r[m].sc.z, sh);
            sc[m][3] = kq_align2(r[m].sc_tail, r[m].sc.w, sh);
            if (!r[m].sh) {
                sc[m][0] = r[m].sc.x;
                sc[m][1] = r[m].sc.y;
                sc[m][2] = r[m].sc.z;
                sc[m][3] = r[m].sc.w;
            }
        }
        const h2 bias = h2{(_Float16)-1056.0f, (_Float16)-1056.0f}; /* 1024 + 32 */
        const _Float16 *xh = st.xh + i * S::kPitch + 256u * b + 4u * g;
        const _Float16 *xl = st.xl + i * S::kPitch + 256u * b + 4u * g;
#pragma unroll
        for (uint32_t nh = 0; nh < 4u; ++nh) {
            const uint32_t n = nh >> 1, h = nh & 1u;
            uint32_t c[NMAT][4];
#pragma unroll
            for (int m = 0; m < NMAT; ++m) {
                const uint32_t A = kq_align2(r[m].w[nh][0].y, r[m].w[nh][0].x, r[m].sh);
                const uint32_t B = kq_align2(r[m].w[nh][1].y, r[m].w[nh][1].x, r[m].sh);
                const uint32_t H = kq_align2(r[m].w[nh][2].y, r[m].w[nh][2].x, r[m].sh);
                c[m][0] = (A & 0x0f0f0f0fu) | ((H << 4) & 0x30303030u);
                c[m][1] = (B & 0x0f0f0f0fu) | ((H << 2) & 0x30303030u);
                c[m][2] = ((A >> 4) & 0x0f0f0f0fu) | (H & 0x30303030u);
                c[m][3] = ((B >> 4) & 0x0f0f0f0fu) | ((H >> 2) & 0x30303030u);
            }
#pragma unroll
            for (uint32_t q = 0; q < 4u; ++q) {
                const uint32_t s = 8u * n + 2u * q + h;
                const uint32_t ko = 128u * n + 32u * q + 16u * h;
                const h4 ah = *(const h4 *)(xh + ko);
                const h4 al = *(const h4 *)(xl + ko);
#pragma unroll
                for (int m = 0; m < NMAT; ++m) {
                    const h2 w0 = bytes_lo(c[m][q]) + bias, w1 = bytes_hi(c[m][q]) + bias;
                    const h4 bw = h4{w0.x, w0.y, w1.x, w1.y};
                    f4 t = {0.f, 0.f, 0.f, 0.f};
                    t = __builtin_amdgcn_mfma_f32_16x16x16f16(ah, bw, t, 0, 0, 0);
                    t = __builtin_amdgcn_mfma_f32_16x16x16f16(al, bw, t, 0, 0, 0);
                    const int8_t scv = (int8_t)((sc[m][s >> 2] >> (8u * (s & 3u))) & 0xffu);
                    const float ds = d[m] * (float)scv;
#pragma unroll
                    for (int k = 0; k < 4; ++k) acc[m][k] = fmaf(ds, t[k], acc[m][k]);
                }
            }
            /* as in the Q4_K tile: bound how far fragment reads are hoisted */
            __builtin_amdgcn_sched_barrier(0);
        }
    }
};

template <uint32_t KSL, int NMAT>
struct Tile<KQ_LAUNCH_Q8_0, KSL, NMAT> {
    using F = Fmt<KQ_LAUNCH_Q8_0>;
    using S = Stage<KQ_LAUNCH_Q8_0, KSL>;
    using Raw = F::Raw;

    /* iteration b: blocks 2b, 2b + 1 of the slice, one step each; the
     * int8 codes enter as fp16 through the offset-binary byte (q + 128) */
    __device__ static __forceinline__ void block(const Raw (&r)[NMAT], const S &st, uint32_t b,
                                                 uint32_t i, uint32_t g, f4 (&acc)[NMAT],
                                                 bool &malformed) {
        const _Float16 *xh = st.xh + i * S::kPitch + 64u * b + 8u * g;
        const _Float16 *xl = st.xl + i * S::kPitch + 64u * b + 8u * g;
        const h2 bias = h2{(_Float16)-1152.0f, (_Float16)-1152.0f}; /* 1024 + 128 */
#pragma unroll
        for (uint32_t bb = 0; bb < 2u; ++bb) {
            const h8 ah = *(const h8 *)(xh + 32u * bb);
            const h8 al = *(const h8 *)(xl + 32u * bb);
#pragma unroll
            for (int m = 0; m < NMAT; ++m) {
                const kq_u32x3 wv = r[m].c[bb];
                /* codes start 2 bytes into the window of even blocks */
                uint32_t c0 = (bb & 1u) ? wv.x : kq_align2(wv.y, wv.x, 2u);
                uint32_t c1 = (bb & 1u) ? wv.y : kq_align2(wv.z, wv.y, 2u);
                c0 ^= 0x80808080u;
                c1 ^= 0x80808080u;
                const h2 w0 = bytes_lo(c0) + bias, w1 = bytes_hi(c0) + bias;
                const h2 w2 = bytes_lo(c1) + bias, w3 = bytes_hi(c1) + bias;
                const h8 bw = h8{w0.x, w0.y, w1.x, w1.y, w2.x, w2.y, w3.x, w3.y};
                f4 t = {0.f, 0.f, 0.f, 0.f};
                t = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bw, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bw, t, 0, 0, 0);
                const float d = half_bits((bb & 1u) ? r[m].d[bb] >> 16 : r[m].d[bb]);
                malformed |= !kq_isfinite(d);
#pragma unroll
                for (int k = 0; k < 4; ++k) acc[m][k] = fmaf(d, t[k], acc[m][k]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
};

template <uint32_t KSL, int NMAT>
struct Tile<KQ_LAUNCH_Q5_1, KSL, NMAT> {
    using F = Fmt<KQ_LAUNCH_Q5_1>;
    using S = Stage<KQ_LAUNCH_Q5_1, KSL>;
    using Raw = F::Raw;

    /* iteration b: blocks 4b .. 4b + 3 of the slice; codes 0..31 are
     * exact in fp16, d scales the step and m the block's activation sum */
    __device__ static __forceinline__ void block(const Raw (&r)[NMAT], const S &st, uint32_t b,
                                                 uint32_t i, uint32_t g, f4 (&acc)[NMAT],
                                                 bool &malformed) {
        const _Float16 *xh = st.xh + i * S::kPitch + 128u * b + 8u * g;
        const _Float16 *xl = st.xl + i * S::kPitch + 128u * b + 8u * g;
        const h2 bias = h2{(_Float16)-1024.0f, (_Float16)-1024.0f};
#pragma unroll
        for (uint32_t bb = 0; bb < 4u; ++bb) {
            const h8 ah = *(const h8 *)(xh + 32u * bb);
            const h8 al = *(const h8 *)(xl + 32u * bb);
            /* this lane's four tokens' sums of the block (times 2^-5) */
            float sx[4];
#pragma unroll
            for (uint32_t q = 0; q < 4u; ++q) {
                const uint32_t so = (4u * g + q) * S::kSxPitch + 4u * b + bb;
                sx[q] = (float)st.sxh[so] + (float)st.sxl[so];
            }
#pragma unroll
            for (int m = 0; m < NMAT; ++m) {
                const kq_u32x2 qv = r[m].q[bb];
                const uint32_t shn = g >= 2u ? 4u : 0u;
                const uint32_t hb = (r[m].qh[bb] >> (8u * g)) & 0xffu;
                const uint32_t c0 = ((qv.x >> shn) & 0x0f0f0f0fu) | spread4(hb & 15u);
                const uint32_t c1 = ((qv.y >> shn) & 0x0f0f0f0fu) | spread4(hb >> 4);
                const h2 w0 = bytes_lo(c0) + bias, w1 = bytes_hi(c0) + bias;
                const h2 w2 = bytes_lo(c1) + bias, w3 = bytes_hi(c1) + bias;
                const h8 bw = h8{w0.x, w0.y, w1.x, w1.y, w2.x, w2.y, w3.x, w3.y};
                f4 t = {0.f, 0.f, 0.f, 0.f};
                t = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bw, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bw, t, 0, 0, 0);
                const float d = half_bits(r[m].dm[bb]), mn = half_bits(r[m].dm[bb] >> 16);
                malformed |= !kq_isfinite(d) || !kq_isfinite(mn);
                const float m32 = mn * 32.0f; /* the sums carry 2^-5 */
#pragma unroll
                for (int k = 0; k < 4; ++k) acc[m][k] = fmaf(d, t[k], fmaf(m32, sx[k], acc[m][k]));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
};

/* ------------------------------------------------------------------ */
/* grouped expert pass */

/* Who a workgroup serves: a routed expert (its tokens at positions
 * offsets[e] .. offsets[e+1]) or a range of 16-token chunks of the shared
 * expert (every token, positions T*K + t). */
struct Work {
    uint32_t first;  /* first position (routed) or first token (shared) */
    uint32_t count;  /* tokens */
    bool shared;
};

__device__ __forceinline__ Work work_of(uint32_t y, const uint32_t *offsets, uint32_t experts,
                                        uint32_t tokens, uint32_t shared_chunks) {
    Work w;
    if (y < experts) {
        w.first = offsets[y];
        w.count = offsets[y + 1u] - w.first;
        w.shared = false;
    } else {
        const uint32_t t0 = (y - experts) * shared_chunks * kTile;
        w.first = t0;
        w.count = t0 < tokens ? min(tokens - t0, shared_chunks * kTile) : 0u;
        w.shared = true;
    }
    return w;
}

/*
 * NMAT = 2: gate and up (rows = routed/shared intermediate, KDIM = hidden),
 *   input rows are the hidden states of the tokens, output act[pos][row] =
 *   swiglu(g, u).
 * NMAT = 1: down (rows = hidden, KDIM = intermediate), input rows are
 *   act[pos], output o[pos][row].
 * grid: x = slabs of NW * TPW * 16 rows, y = routed experts then shared
 * chunks. Positions: routed pairs 0 .. T*K-1 (permuted order), shared token
 * t at T*K + t.
 *
 * Each wave walks TPW 16-row tiles, all blocks of a tile in order, with the
 * next block's weights (across tile boundaries) in flight while one block is
 * multiplied. Every prefetch and every result store is issued on every
 * path -- ones past the data use offsets outside their buffer, which the
 * hardware drops -- so the memory counters the compiler waits on are the
 * same on every path and a wait never drains the prefetch.
 */
template <uint32_t GFMT, uint32_t KDIM, int NMAT, int NW, int TPW, int PD, int KS>
__global__ __launch_bounds__(NW * 64) void grouped_pass(
    const uint8_t *__restrict__ W0, const uint8_t *__restrict__ W1,
    const uint8_t *__restrict__ SW0, const uint8_t *__restrict__ SW1,
    const float *__restrict__ X, const uint32_t *__restrict__ offsets,
    const uint32_t *__restrict__ perm_tok, uint32_t experts, uint32_t tokens, uint32_t top_k,
    uint32_t rows, uint32_t shared_chunks, uint32_t ybase, float *__restrict__ out,
    uint32_t *status) {
    /* KS slices of KSL columns: the activation image of one slice is staged
     * at a time (a 2560-column image would not fit the LDS); the
     * accumulators carry over (one tile per wave then) */
    constexpr uint32_t KSL = KDIM / (uint32_t)KS;
    static_assert(KS == 1 || TPW == 1, "sliced passes run one tile per wave");
    using F = Fmt<GFMT>;
    using S = Stage<GFMT, KSL>;
    using T = Tile<GFMT, KSL, NMAT>;
    using Raw = typename F::Raw;
    constexpr uint32_t NB = KDIM / F::kUnit;       /* units of a row */
    constexpr uint32_t NBS = NB / (uint32_t)KS;    /* units of a slice */
    static_assert(NBS * (uint32_t)KS == NB && NB * F::kUnit == KDIM, "whole units per slice");
    constexpr uint32_t RB = NB * F::kUnitBytes;
    __shared__ S st;
    __shared__ int src_row[kTile];

    const uint32_t e = blockIdx.y + ybase;
    const Work wk = work_of(e, offsets, experts, tokens, shared_chunks);
    if (wk.count == 0u) return;
    /* the wave index is uniform across the wave; saying so keeps the weight
     * buffer descriptors in scalar registers (no per-lane waterfall) */
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 15u, g = lane >> 4;
    const uint32_t tk = tokens * top_k;
    /* tile t of this wave starts at row tile_row(t); tiles past the matrix
     * load nothing and store nothing */
    auto tile_row = [&](uint32_t t) { return ((blockIdx.x * TPW + t) * NW + wave) * kTile; };

    const uint32_t wbytes = rows * RB;
    KqBuf wb[NMAT];
#pragma unroll
    for (int m = 0; m < NMAT; ++m) {
        const uint8_t *base = wk.shared ? (m == 0 ? SW0 : SW1)
                                        : (m == 0 ? W0 : W1) + (size_t)e * rows * RB;
        wb[m] = kq_buf(base, wbytes);
    }
    /* byte offset of unit u of tile t for this lane's row, or the buffer
     * size (every field read from there is dropped) */
    auto boff = [&](uint32_t t, uint32_t u) {
        const uint32_t r0 = tile_row(t);
        return (t < (uint32_t)TPW && r0 < rows) ? (r0 + j) * RB + u * F::kUnitBytes : wbytes;
    };
    auto load = [&](Raw (&r)[NMAT], uint32_t off) {
#pragma unroll
        for (int m = 0; m < NMAT; ++m) r[m] = F::load(wb[m], off, g);
    };
    /* results go through a buffer over this workgroup's output rows */
    const uint32_t pos0 = wk.shared ? tk + wk.first : wk.first;
    const uint32_t obytes = wk.count * rows * 4u;
    const KqBuf ob = kq_buf(out + (size_t)pos0 * rows, obytes);

    /* the wave's iterations are (slice, tile, unit of the slice) in order;
     * iteration `it` reads ring slot it % R, which iteration it - PD filled */
    constexpr uint32_t PER = (uint32_t)TPW * NBS; /* iterations per slice */
    constexpr uint32_t NIT = (uint32_t)KS * PER;
    constexpr uint32_t R = (uint32_t)PD + 1u;
    auto it_off = [&](uint32_t it) {
        if (it >= NIT) return wbytes;
        const uint32_t ks = it / PER, rem = it % PER;
        return boff(rem / NBS, ks * NBS + rem % NBS);
    };

    bool bad = false, badin = false, malformed = false;
    auto stage = [&](uint32_t ks) {
        /* a non-finite hidden state is the caller's input; a non-finite
         * intermediate activation is a numeric failure of the layer */
        const bool nf = stage_slice<GFMT, KDIM, KSL>(st, X, ks * KSL, src_row, wave, NW, lane);
        if (NMAT == 2)
            badin |= nf;
        else
            bad |= nf;
    };
    for (uint32_t c0 = 0; c0 < wk.count; c0 += kTile) {
        /* the first PD units' weights are requested before the staging */
        Raw ring[R][NMAT];
#pragma unroll
        for (uint32_t it = 0; it < (uint32_t)PD; ++it) load(ring[it], it_off(it));
        __syncthreads(); /* the previous chunk's readers are done */
        if (threadIdx.x < kTile) {
            const uint32_t i = threadIdx.x;
            int src = -1;
            if (c0 + i < wk.count) {
                const uint32_t p = wk.first + c0 + i;
                if (NMAT == 2)
                    src = (int)(wk.shared ? p : perm_tok[p]);
                else
                    src = (int)(wk.shared ? tk + p : p);
            }
            src_row[i] = src;
        }
        __syncthreads();
        stage(0u);
        __syncthreads();

        f4 acc[NMAT];
        static_assert(NIT % R == 0u, "the ring must divide the iterations");
#pragma unroll 1
        for (uint32_t it0 = 0; it0 < NIT; it0 += R) {
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                const uint32_t it = it0 + r;
                const uint32_t ks = it / PER, rem = it % PER;
                const uint32_t t = rem / NBS, b = rem % NBS;
                if (KS > 1 && ks > 0u && rem == 0u) {
                    /* the next slice of the activations */
                    __syncthreads();
                    stage(ks);
                    __syncthreads();
                }
                if (b == 0u && ks == 0u) {
#pragma unroll
                    for (int m = 0; m < NMAT; ++m) acc[m] = f4{0.f, 0.f, 0.f, 0.f};
                }
                load(ring[(r + PD) % R], it_off(it + PD));
                T::block(ring[r], st, b, j, g, acc, malformed);
                __builtin_amdgcn_sched_barrier(0);
                if (b + 1u < NBS || ks + 1u < (uint32_t)KS) continue;
                /* D[token][row]: this lane holds row `row` of tokens 4g .. 4g+3 */
                const uint32_t row = tile_row(t) + j;
#pragma unroll
                for (uint32_t q = 0; q < 4u; ++q) {
                    const uint32_t i = 4u * g + q;
                    const bool valid = c0 + i < wk.count && row < rows;
                    const int sg = st.sig[i];
                    float v;
                    if constexpr (NMAT == 2) {
                        const float gv = ldexpf(acc[0][q], -sg), uv = ldexpf(acc[1][q], -sg);
                        v = kq_swiglu(gv, uv);
                        bad |= valid && (!kq_isfinite(gv) || !kq_isfinite(uv));
                    } else {
                        v = ldexpf(acc[0][q], -sg);
                    }
                    bad |= valid && !kq_isfinite(v);
                    const uint32_t off = valid ? ((c0 + i) * rows + row) * 4u : obytes;
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), ob.r, (int)off, 0,
                                                          0);
                }
            }
        }
    }
    if (badin) kq_flag(status, KQ_DEV_INPUT);
    if (malformed) kq_flag(status, KQ_DEV_MALFORMED);
    if (bad) kq_flag(status, KQ_DEV_NUMERIC);
}

/* ------------------------------------------------------------------ */
/* permutation: stable counting sort of (token, slot) pairs by expert id */

constexpr uint32_t kPermChunk = 256; /* tokens per rank pass */

/* The Q4_K gate/up pass's work list (kq_grouped_gu.hip, gu_items): one
 * item per item_rows-token chunk of an expert, routed experts in id order,
 * then the shared expert's chunks; [0] the count, items from [4] on as
 * (expert | kItemShared, first | count << 24). */
constexpr uint32_t kItemRows = 16;     /* of the 16-token passes */
constexpr uint32_t kWideItemRows = 64; /* of kq_gemm.hip */
constexpr uint32_t kItemShared = 0x80000000u;

__global__ __launch_bounds__(1024) void moe_permute(const uint32_t *__restrict__ ids,
                                                    uint32_t tokens, uint32_t top_k,
                                                    uint32_t experts, uint32_t *__restrict__ offsets,
                                                    uint32_t *__restrict__ perm_tok,
                                                    uint32_t *__restrict__ pos,
                                                    uint32_t *__restrict__ pair_slot,
                                                    uint32_t *status, uint32_t *items,
                                                    uint32_t with_shared, uint32_t item_rows,
                                                    uint32_t *zero, uint32_t nzero) {
    __shared__ uint32_t cnt[1024];
    __shared__ uint32_t base[1024];
    __shared__ uint32_t bits[1024][kPermChunk / 32u];
    __shared__ uint32_t wsum[16];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const uint32_t pairs = tokens * top_k;
    cnt[tid] = 0u;
    /* words a later pass accumulates into (atomic maxima) start at zero */
    for (uint32_t i = tid; i < nzero; i += 1024u) zero[i] = 0u;
    __syncthreads();
    bool bad = false;
    for (uint32_t p = tid; p < pairs; p += 1024u) {
        uint32_t e = ids[p];
        if (e >= experts) {
            bad = true;
            e = 0u;
        }
        atomicAdd(&cnt[e], 1u);
    }
    __syncthreads();
    /* exclusive scan of cnt[0 .. 1023] (entries past the experts are 0) */
    {
        const uint32_t v = cnt[tid];
        uint32_t incl = v;
#pragma unroll
        for (uint32_t o = 1; o < 64u; o <<= 1) {
            const uint32_t n = __shfl_up(incl, o, KQ_WAVE);
            if (lane >= o) incl += n;
        }
        if (lane == 63u) wsum[wave] = incl;
        __syncthreads();
        uint32_t before = 0u;
        for (uint32_t w = 0; w < wave; ++w) before += wsum[w];
        const uint32_t ex = before + incl - v;
        base[tid] = ex;
        if (tid < experts) offsets[tid] = ex;
        if (tid == experts) offsets[tid] = ex; /* = pairs */
    }
    __syncthreads();
    if (items != nullptr) {
        /* the gate/up work list from the same counts: exclusive scan of
         * the chunks per expert */
        __shared__ uint32_t csum[16];
        const uint32_t c = tid < experts ? cnt[tid] : 0u;
        const uint32_t nc = (c + item_rows - 1u) / item_rows;
        uint32_t incl = nc;
#pragma unroll
        for (uint32_t o = 1; o < 64u; o <<= 1) {
            const uint32_t n = __shfl_up(incl, o, KQ_WAVE);
            if (lane >= o) incl += n;
        }
        if (lane == 63u) csum[wave] = incl;
        __syncthreads();
        uint32_t ib = incl - nc, total = 0u;
        for (uint32_t w = 0; w < 16u; ++w) {
            ib += w < wave ? csum[w] : 0u;
            total += csum[w];
        }
        uint32_t *list = items + 4;
        const uint32_t o0 = base[tid];
        for (uint32_t k = 0; k < nc; ++k) {
            list[2u * (ib + k)] = tid;
            list[2u * (ib + k) + 1u] = (o0 + item_rows * k) | (min(c - item_rows * k, item_rows) << 24);
        }
        const uint32_t nsh = with_shared ? (tokens + item_rows - 1u) / item_rows : 0u;
        for (uint32_t k = tid; k < nsh; k += 1024u) {
            list[2u * (total + k)] = kItemShared | k;
            list[2u * (total + k) + 1u] = (item_rows * k) | (min(tokens - item_rows * k, item_rows) << 24);
        }
        if (tid == 0u) items[0] = total + nsh;
    }
    for (uint32_t t0 = 0; t0 < tokens; t0 += kPermChunk) {
        const uint32_t nt = min(kPermChunk, tokens - t0);
        for (uint32_t w = tid; w < 1024u * (kPermChunk / 32u); w += 1024u)
            (&bits[0][0])[w] = 0u;
        __syncthreads();
        const uint32_t np = nt * top_k;
        for (uint32_t p = tid; p < np; p += 1024u) {
            const uint32_t lt = p / top_k;
            uint32_t e = ids[(size_t)t0 * top_k + p];
            e = e < experts ? e : 0u;
            atomicOr(&bits[e][lt >> 5], 1u << (lt & 31u));
        }
        __syncthreads();
        for (uint32_t p = tid; p < np; p += 1024u) {
            const uint32_t lt = p / top_k;
            uint32_t e = ids[(size_t)t0 * top_k + p];
            e = e < experts ? e : 0u;
            uint32_t r = __popc(bits[e][lt >> 5] & ((1u << (lt & 31u)) - 1u));
            for (uint32_t w = 0; w < (lt >> 5); ++w) r += __popc(bits[e][w]);
            const uint32_t q = base[e] + r;
            pos[(size_t)t0 * top_k + p] = q;
            perm_tok[q] = t0 + lt;
            if (pair_slot != nullptr) pair_slot[q] = p - lt * top_k;
        }
        __syncthreads();
        {
            uint32_t c = 0u;
#pragma unroll
            for (uint32_t w = 0; w < kPermChunk / 32u; ++w) c += __popc(bits[tid][w]);
            base[tid] += c;
        }
        __syncthreads();
    }
    if (bad) kq_flag(status, KQ_DEV_RANGE);
}

/* ------------------------------------------------------------------ */
/* combine, in the reference's order (src/kq_moe_qwen38.c:722-765, :826) */

/* One thread per four consecutive outputs of a token: the slots' rows are
 * requested together (up to kCombineRun of them before the first add),
 * then summed in the reference's order with separately rounded products. */
constexpr uint32_t kCombineRun = 16;

__global__ __launch_bounds__(256) void moe_combine(
    const float *__restrict__ o, const uint32_t *__restrict__ pos,
    const uint32_t *__restrict__ order, const float *__restrict__ weights,
    const float *__restrict__ shared_scale, uint32_t tokens, uint32_t top_k, uint32_t hidden,
    float *__restrict__ out, uint32_t *status) {
    const uint32_t t = blockIdx.y;
    const uint32_t q = blockIdx.x * 256u + threadIdx.x; /* float4 of the row */
    const uint32_t hq = hidden / 4u;
    if (q >= hq) return;
    const uint32_t tk = tokens * top_k;
    const float4 *o4 = (const float4 *)o;
    bool bad = false;
    float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
    auto add = [&](const float4 v, const float w) {
        bad |= !kq_isfinite(v.x) || !kq_isfinite(v.y) || !kq_isfinite(v.z) || !kq_isfinite(v.w);
        float p;
        p = v.x * w; sum.x = sum.x + p;
        p = v.y * w; sum.y = sum.y + p;
        p = v.z * w; sum.z = sum.z + p;
        p = v.w * w; sum.w = sum.w + p;
    };
    for (uint32_t j0 = 0; j0 < top_k; j0 += kCombineRun) {
        float4 v[kCombineRun];
        float wv[kCombineRun];
#pragma unroll
        for (uint32_t i = 0; i < kCombineRun; ++i) {
            if (j0 + i < top_k) {
                const uint32_t sl = order[(size_t)t * top_k + j0 + i];
                const uint32_t p = pos[(size_t)t * top_k + sl];
                wv[i] = weights[(size_t)t * top_k + sl];
                v[i] = o4[(size_t)p * hq + q];
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < kCombineRun; ++i)
            if (j0 + i < top_k) add(v[i], wv[i]);
    }
    const float4 so = o4[(size_t)(tk + t) * hq + q];
    const float sc = shared_scale[t];
    float4 r;
    auto fin = [&](float sv, float sm, float &dst) {
        const float gated = sv * sc;
        const float val = sm + gated;
        bad |= !kq_isfinite(sv) || !kq_isfinite(sm) || !kq_isfinite(gated) || !kq_isfinite(val);
        dst = val;
    };
    fin(so.x, sum.x, r.x);
    fin(so.y, sum.y, r.y);
    fin(so.z, sum.z, r.z);
    fin(so.w, sum.w, r.w);
    ((float4 *)out)[(size_t)t * hq + q] = r;
    if (bad) kq_flag(status, KQ_DEV_NUMERIC);
}

/* ------------------------------------------------------------------ */
/* launchers */

constexpr uint32_t kSharedChunks = 2; /* 16-token chunks per shared-expert workgroup */

/* Launch shape per pass: NW waves per workgroup, TPW 16-row tiles per
 * wave, PD blocks of weights in flight ahead of the one being multiplied.
 * The registers of a SIMD bound waves x (PD + 1) x block registers; the
 * gate/up image (136 KiB at 2048 columns) allows one workgroup per CU. */
#ifndef KQ_GU_NW
#define KQ_GU_NW 16
#define KQ_GU_TPW 1
#define KQ_GU_PD 1
#endif
#ifndef KQ_DN_NW
#define KQ_DN_NW 8
#define KQ_DN_TPW 4
#define KQ_DN_PD 1
#endif
#ifndef KQ_GU_KSL
#define KQ_GU_KSL 2048 /* widest activation slice staged at once */
#endif

/* slices of a row: the fewest whole-unit slices of at most KQ_GU_KSL
 * columns */
template <uint32_t GFMT, uint32_t KDIM>
constexpr int gu_slices() {
    for (int ks = 1; ks <= 16; ++ks) {
        const uint32_t w = KDIM / (uint32_t)ks;
        if (w * (uint32_t)ks == KDIM && w % Fmt<GFMT>::kUnit == 0u && w <= (uint32_t)KQ_GU_KSL)
            return ks;
    }
    return 0;
}
template <uint32_t GFMT, uint32_t KDIM, int NMAT>
struct Shape {
    /* rows longer than KQ_GU_KSL columns are staged in slices, one tile
     * per wave */
    static constexpr bool kSliced = KDIM > (uint32_t)KQ_GU_KSL;
    static constexpr int NW = NMAT == 2 ? (KDIM >= 1024u ? KQ_GU_NW : 8)
                                        : (kSliced ? KQ_GU_NW : KQ_DN_NW);
    static constexpr int TPW = NMAT == 2 ? (KDIM >= 1024u ? KQ_GU_TPW : 2)
                                         : (kSliced ? 1 : KQ_DN_TPW);
    static constexpr int KS = gu_slices<GFMT, KDIM>();
    static_assert(KS >= 1, "no slicing of this row length");
    static_assert(KS == 1 || TPW == 1, "sliced passes run one tile per wave");
    /* the ring (PD + 1 slots) is a power of two that divides the wave's
     * KS * TPW * KDIM / unit iterations */
    static constexpr int NIT = TPW * (int)(KDIM / Fmt<GFMT>::kUnit);
    static constexpr int WANT = (NMAT == 2 ? KQ_GU_PD : KQ_DN_PD) + 1;
    static constexpr int RING = WANT >= 8 && NIT % 8 == 0 ? 8
                                : WANT >= 4 && NIT % 4 == 0 ? 4
                                : WANT >= 2 && NIT % 2 == 0 ? 2 : 1;
    static constexpr int PD = RING > 1 ? RING - 1 : 0;
};

/* the Q6_K down pass with its weights streamed through LDS (below) */
template <uint32_t KDIM>
hipError_t launch_down_q6k(const uint8_t *W0, const uint8_t *SW0, const float *X,
                           const uint32_t *offsets, uint32_t experts, uint32_t tokens,
                           uint32_t top_k, uint32_t rows, uint32_t y0, uint32_t ny,
                           uint32_t chunks, float *out, uint32_t *status, hipStream_t s);

/* Workgroup rows y0 .. y0 + ny - 1 of the pass: experts 0 .. E-1, then the
 * shared expert's chunk groups. */
template <uint32_t GFMT, uint32_t KDIM, int NMAT>
hipError_t launch_pass(const uint8_t *W0, const uint8_t *W1, const uint8_t *SW0,
                       const uint8_t *SW1, const float *X, const uint32_t *offsets,
                       const uint32_t *perm_tok, uint32_t experts, uint32_t tokens,
                       uint32_t top_k, uint32_t rows, uint32_t y0, uint32_t ny, uint32_t chunks,
                       float *out, uint32_t *status, hipStream_t s) {
    if (ny == 0u) return hipSuccess;
    /* (an intermediate of 2048 leaves no LDS beside its activation image
     * for the weight slots) */
    if constexpr (GFMT == KQ_LAUNCH_Q6_K && NMAT == 1 && KDIM <= 1024u)
        return launch_down_q6k<KDIM>(W0, SW0, X, offsets, experts, tokens, top_k, rows, y0, ny,
                                     chunks, out, status, s);
    constexpr int NW = Shape<GFMT, KDIM, NMAT>::NW;
    constexpr int TPW = Shape<GFMT, KDIM, NMAT>::TPW;
    constexpr int PD = Shape<GFMT, KDIM, NMAT>::PD;
    constexpr int KS = Shape<GFMT, KDIM, NMAT>::KS;
    if (y0 >= experts && ny > 0u) {
        /* the shared expert alone (its format differs from the routed
         * one): a few rows for every token, so 64-row slabs and one
         * 16-token chunk per workgroup, which spreads it over the device */
        constexpr int NWS = 4;
        /* the ring (a power of two) must divide the TPW = 1 iterations */
        constexpr int NIT1 = (int)(KDIM / Fmt<GFMT>::kUnit);
        constexpr int R1 = (PD + 1) >= 8 && NIT1 % 8 == 0   ? 8
                           : (PD + 1) >= 4 && NIT1 % 4 == 0 ? 4
                           : (PD + 1) >= 2 && NIT1 % 2 == 0 ? 2
                                                            : 1;
        constexpr int PD1 = R1 - 1;
        const uint32_t nys = (tokens + kTile - 1u) / kTile;
        const dim3 grid((rows + NWS * kTile - 1u) / (NWS * kTile), nys);
        hipLaunchKernelGGL((grouped_pass<GFMT, KDIM, NMAT, NWS, 1, PD1, KS>), grid,
                           dim3(NWS * 64), 0, s, W0, W1, SW0, SW1, X, offsets, perm_tok, experts,
                           tokens, top_k, rows, 1u, y0, out, status);
        return hipGetLastError();
    }
    const uint32_t slab = (uint32_t)(NW * TPW) * kTile;
    const dim3 grid((rows + slab - 1u) / slab, ny);
    hipLaunchKernelGGL((grouped_pass<GFMT, KDIM, NMAT, NW, TPW, PD, KS>), grid, dim3(NW * 64), 0,
                       s, W0, W1, SW0, SW1, X, offsets, perm_tok, experts, tokens, top_k, rows,
                       chunks, y0, out, status);
    return hipGetLastError();
}

/* the row lengths each format's pass is built for: whole units, and the
 * activation image of a slice within the LDS */
template <uint32_t GFMT, int NMAT>
constexpr bool pass_dim(uint32_t k) {
    if (k % Fmt<GFMT>::kUnit != 0u) return false;
    if (NMAT == 2) return k == 256u || k == 512u || k == 1024u || k == 2048u || k == 2560u;
    return k == 256u || k == 320u || k == 512u || k == 640u || k == 1024u || k == 2048u ||
           k == 10240u;
}

template <uint32_t GFMT, int NMAT>
hipError_t pass_cols(uint32_t kdim, const uint8_t *W0, const uint8_t *W1, const uint8_t *SW0,
                     const uint8_t *SW1, const float *X, const uint32_t *offsets,
                     const uint32_t *perm_tok, uint32_t experts, uint32_t tokens, uint32_t top_k,
                     uint32_t rows, uint32_t y0, uint32_t ny, uint32_t chunks, float *out,
                     uint32_t *status, hipStream_t s) {
#define KQ_PASS(K)                                                                               \
    if constexpr (pass_dim<GFMT, NMAT>(K))                                                       \
        return launch_pass<GFMT, K, NMAT>(W0, W1, SW0, SW1, X, offsets, perm_tok, experts,       \
                                          tokens, top_k, rows, y0, ny, chunks, out, status, s);  \
    return hipErrorInvalidValue
    switch (kdim) {
    case 256: { KQ_PASS(256u); }
    case 320: { KQ_PASS(320u); }
    case 512: { KQ_PASS(512u); }
    case 640: { KQ_PASS(640u); }
    case 1024: { KQ_PASS(1024u); }
    case 2048: { KQ_PASS(2048u); }
    case 2560: { KQ_PASS(2560u); }
    case 10240: { KQ_PASS(10240u); }
    default: return hipErrorInvalidValue;
    }
#undef KQ_PASS
}

/* pass_dim for a run-time format */
bool pass_dim_rt(uint32_t type, int nmat, uint32_t k) {
    switch (type) {
    case KQ_LAUNCH_Q4_K: return nmat == 2 ? pass_dim<KQ_LAUNCH_Q4_K, 2>(k) : pass_dim<KQ_LAUNCH_Q4_K, 1>(k);
    case KQ_LAUNCH_Q6_K: return nmat == 1 && pass_dim<KQ_LAUNCH_Q6_K, 1>(k);
    case KQ_LAUNCH_Q8_0: return nmat == 2 ? pass_dim<KQ_LAUNCH_Q8_0, 2>(k) : pass_dim<KQ_LAUNCH_Q8_0, 1>(k);
    case KQ_LAUNCH_Q5_1: return nmat == 1 && pass_dim<KQ_LAUNCH_Q5_1, 1>(k);
    default: return false;
    }
}

/* one pass of a role whose routed and shared matrices may differ in
 * format: one launch when they agree, else the routed workgroups and the
 * shared ones as two launches */
template <int NMAT>
hipError_t pass_any(uint32_t type, uint32_t kdim, const uint8_t *W0, const uint8_t *W1,
                    const uint8_t *SW0, const uint8_t *SW1, const float *X,
                    const uint32_t *offsets, const uint32_t *perm_tok, uint32_t experts,
                    uint32_t tokens, uint32_t top_k, uint32_t rows, uint32_t y0, uint32_t ny,
                    float *out, uint32_t *status, hipStream_t s) {
#define KQ_ANY(F)                                                                              \
    pass_cols<F, NMAT>(kdim, W0, W1, SW0, SW1, X, offsets, perm_tok, experts, tokens, top_k, \
                       rows, y0, ny, kSharedChunks, out, status, s)
    switch (type) {
    case KQ_LAUNCH_Q4_K: return KQ_ANY(KQ_LAUNCH_Q4_K);
    case KQ_LAUNCH_Q8_0: return KQ_ANY(KQ_LAUNCH_Q8_0);
    case KQ_LAUNCH_Q6_K:
        if constexpr (NMAT == 1) return KQ_ANY(KQ_LAUNCH_Q6_K);
        return hipErrorInvalidValue;
    case KQ_LAUNCH_Q5_1:
        if constexpr (NMAT == 1) return KQ_ANY(KQ_LAUNCH_Q5_1);
        return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
    }
#undef KQ_ANY
}

/* ------------------------------------------------------------------ */
/* one 256-column Q6_K block of 16 rows in LDS: 224-byte windows (a block
 * from its 4-byte aligned start) at a 240-byte pitch, so lanes (row, k-group)
 * hit distinct banks */
constexpr uint32_t kMvWin = 224u;
constexpr uint32_t kMvPitch = 240u;
constexpr uint32_t kMvSlot = kTile * kMvPitch;
constexpr uint32_t kMvUnits = kTile * (kMvWin / 16u);   /* 16-byte loads per block: 224 */
constexpr int kMvLoads = (int)((kMvUnits + 63u) / 64u); /* per lane: 4 */

/* ------------------------------------------------------------------ */
/* grouped Q6_K down pass with its weights streamed through LDS
 *
 * The same work split, staging and Tile<Q6_K> steps as grouped_pass, but
 * the block operand pieces (twelve scattered 4-byte windows per lane) are
 * not fetched from global memory: each wave loads one 16-row block of its
 * tile contiguously into a private LDS slot, two
 * blocks ahead of the one it multiplies, and the Raw pieces are read from
 * there. Offsets past the matrix read as zeros and stores past the
 * workgroup's outputs are dropped, so no path branches around a load. */
template <uint32_t KDIM, int NW, int TPW>
__global__ __launch_bounds__(NW * 64) void grouped_down_q6k(
    const uint8_t *__restrict__ W0, const uint8_t *__restrict__ SW0,
    const float *__restrict__ X, const uint32_t *__restrict__ offsets, uint32_t experts,
    uint32_t tokens, uint32_t top_k, uint32_t rows, uint32_t shared_chunks, uint32_t ybase,
    float *__restrict__ out, uint32_t *status) {
    using F = Fmt<KQ_LAUNCH_Q6_K>;
    using S = Stage<KQ_LAUNCH_Q6_K, KDIM>;
    using T = Tile<KQ_LAUNCH_Q6_K, KDIM, 1>;
    using Raw = F::Raw;
    constexpr uint32_t NB = KDIM / 256u;
    constexpr uint32_t RB = NB * F::kBytes;
    constexpr uint32_t NIT = (uint32_t)TPW * NB;
    static_assert(NIT % 2u == 0u, "items run in pairs");
    __shared__ S st;
    __shared__ int src_row[kTile];
    __shared__ __align__(16) uint8_t slots[NW][2][kMvSlot];

    const uint32_t e = blockIdx.y + ybase;
    const Work wk = work_of(e, offsets, experts, tokens, shared_chunks);
    if (wk.count == 0u) return;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 15u, g = lane >> 4;
    const uint32_t tk = tokens * top_k;
    auto tile_row = [&](uint32_t t) { return ((blockIdx.x * TPW + t) * NW + wave) * kTile; };
    const uint32_t wbytes = rows * RB;
    const KqBuf wb = kq_buf(wk.shared ? SW0 : W0 + (size_t)e * rows * RB, wbytes);
    const uint32_t pos0 = wk.shared ? tk + wk.first : wk.first;
    const uint32_t obytes = wk.count * rows * 4u;
    const KqBuf ob = kq_buf(out + (size_t)pos0 * rows, obytes);
    uint8_t *myslot = &slots[wave][0][0];

    /* item it = block it % NB of tile it / NB; unit e = i * 64 + lane of
     * its 224 loads covers bytes [16u, 16u + 16) of row e / 14's window
     * (the block start rounded down to 4 bytes) */
    typedef kq_u32x4 Ld[kMvLoads];
    auto load_item = [&](uint32_t it, Ld &v) {
        const uint32_t t = it / NB, b = it % NB;
#pragma unroll
        for (int i = 0; i < kMvLoads; ++i) {
            const uint32_t u0 = (uint32_t)i * 64u + lane;
            const uint32_t r = u0 / 14u, u = u0 - 14u * r;
            const uint32_t row = tile_row(t) + r;
            const uint32_t o = row * RB + b * F::kBytes;
            const uint32_t off = (u0 < kMvUnits && t < (uint32_t)TPW && row < rows)
                                     ? (o & ~3u) + 16u * u
                                     : wbytes + 256u;
            v[i] = __builtin_amdgcn_raw_buffer_load_b128(wb.r, (int)off, 0, 0);
        }
    };
    auto store_item = [&](uint32_t slot, const Ld &v) {
#pragma unroll
        for (int i = 0; i < kMvLoads; ++i) {
            const uint32_t u0 = (uint32_t)i * 64u + lane;
            const uint32_t r = u0 / 14u, u = u0 - 14u * r;
            if (u0 < kMvUnits)
                *(kq_u32x4 *)(myslot + slot * kMvSlot + r * kMvPitch + 16u * u) = v[i];
        }
    };
    /* the pieces Fmt<Q6_K>::load would read, from this lane's row in slot */
    auto lds_raw = [&](uint32_t slot, uint32_t t, uint32_t b) {
        const uint32_t o = (tile_row(t) + j) * RB + b * F::kBytes;
        const uint8_t *p = myslot + slot * kMvSlot + j * kMvPitch;
        auto w32 = [&](uint32_t off) { return *(const uint32_t *)(p + off); };
        Raw r;
        r.sh = o & 3u;
#pragma unroll
        for (uint32_t nh = 0; nh < 4u; ++nh) {
            const uint32_t n = nh >> 1, h = nh & 1u;
            const uint32_t oa = 64u * n + 16u * h + 4u * g;
            const uint32_t oq = 128u + 32u * n + 16u * h + 4u * g;
            r.w[nh][0] = kq_u32x2{w32(oa), w32(oa + 4u)};
            r.w[nh][1] = kq_u32x2{w32(oa + 32u), w32(oa + 36u)};
            r.w[nh][2] = kq_u32x2{w32(oq), w32(oq + 4u)};
        }
        r.sc = make_uint4(w32(192u), w32(196u), w32(200u), w32(204u));
        r.sc_tail = w32(208u);
        r.d = *(const uint16_t *)(p + r.sh + 208u);
        return r;
    };

    bool bad = false, malformed = false;
    for (uint32_t c0 = 0; c0 < wk.count; c0 += kTile) {
        Ld va, vb;
        load_item(0u, va);
        load_item(1u, vb);
        __syncthreads(); /* the previous chunk's readers are done */
        if (threadIdx.x < kTile) {
            const uint32_t i = threadIdx.x;
            int src = -1;
            if (c0 + i < wk.count) {
                const uint32_t p = wk.first + c0 + i;
                src = (int)(wk.shared ? tk + p : p);
            }
            src_row[i] = src;
        }
        __syncthreads();
        /* a non-finite intermediate activation is a numeric failure */
        bad |= stage_rows<KQ_LAUNCH_Q6_K, KDIM>(st, X, src_row, wave, NW, lane);
        __syncthreads();
        store_item(0u, va);
        load_item(2u, va);

        f4 acc[1];
        auto process = [&](uint32_t it, uint32_t slot) {
            const uint32_t t = it / NB, b = it % NB;
            if (b == 0u) acc[0] = f4{0.f, 0.f, 0.f, 0.f};
            const Raw rr[1] = {lds_raw(slot, t, b)};
            T::block(rr, st, b, j, g, acc, malformed);
            __builtin_amdgcn_sched_barrier(0);
            if (b + 1u < NB) return;
            /* D[token][row]: this lane holds row `row` of tokens 4g .. 4g+3 */
            const uint32_t row = tile_row(t) + j;
#pragma unroll
            for (uint32_t q = 0; q < 4u; ++q) {
                const uint32_t i = 4u * g + q;
                const bool valid = c0 + i < wk.count && row < rows;
                const float v = ldexpf(acc[0][q], -st.sig[i]);
                bad |= valid && !kq_isfinite(v);
                const uint32_t off = valid ? ((c0 + i) * rows + row) * 4u : obytes;
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), ob.r, (int)off, 0, 0);
            }
        };
#pragma unroll 1
        for (uint32_t it = 0; it < NIT; it += 2u) {
            process(it, 0u);
            store_item(1u, vb);
            load_item(it + 3u, vb);
            process(it + 1u, 1u);
            store_item(0u, va);
            load_item(it + 4u, va);
        }
    }
    if (malformed) kq_flag(status, KQ_DEV_MALFORMED);
    if (bad) kq_flag(status, KQ_DEV_NUMERIC);
}

template <uint32_t KDIM>
hipError_t launch_down_q6k(const uint8_t *W0, const uint8_t *SW0, const float *X,
                           const uint32_t *offsets, uint32_t experts, uint32_t tokens,
                           uint32_t top_k, uint32_t rows, uint32_t y0, uint32_t ny,
                           uint32_t chunks, float *out, uint32_t *status, hipStream_t s) {
    constexpr int NW = Shape<KQ_LAUNCH_Q6_K, KDIM, 1>::NW;
    constexpr int TPW = Shape<KQ_LAUNCH_Q6_K, KDIM, 1>::TPW;
    const uint32_t slab = (uint32_t)(NW * TPW) * kTile;
    const dim3 grid((rows + slab - 1u) / slab, ny);
    hipLaunchKernelGGL((grouped_down_q6k<KDIM, NW, TPW>), grid, dim3(NW * 64), 0, s, W0, SW0, X,
                       offsets, experts, tokens, top_k, rows, chunks, y0, out, status);
    return hipGetLastError();
}

}  // namespace

extern "C" int kq_launch_moe_grouped_supported(const kq_launch_moe_dims *d,
                                               const kq_launch_moe_weights *w) {
    /* gate/up in Q4_K (the 6-bit scales fold into exact fp16 weights) or
     * Q8_0, or Q5_K through the LDS pass (a Q5_K shared expert only with
     * Q5_K routed experts, in the same pass); down in Q4_K, Q6_K, Q5_1 or
     * Q8_0; routed and shared each of their own format, at the row lengths
     * each pass is built for */
    const bool q5 = w->gate_type == KQ_LAUNCH_Q5_K &&
                    kq_launch_gu_lds_supported(KQ_LAUNCH_Q5_K, d->hidden);
    return w->up_type == w->gate_type && w->shared_up_type == w->shared_gate_type &&
           (pass_dim_rt(w->gate_type, 2, d->hidden) || q5) &&
           (pass_dim_rt(w->shared_gate_type, 2, d->hidden) ||
            (q5 && w->shared_gate_type == KQ_LAUNCH_Q5_K)) &&
           pass_dim_rt(w->down_type, 1, d->inter) &&
           pass_dim_rt(w->shared_down_type, 1, d->inter) && d->inter == d->shared_inter &&
           d->experts <= 1023u;
}

extern "C" hipError_t kq_launch_moe_permute(const uint32_t *ids, uint32_t tokens, uint32_t top_k,
                                            uint32_t experts, uint32_t *offsets,
                                            uint32_t *pair_token, uint32_t *pos,
                                            uint32_t *pair_slot, uint32_t *status,
                                            hipStream_t s) {
    hipLaunchKernelGGL(moe_permute, dim3(1), dim3(1024), 0, s, ids, tokens, top_k, experts,
                       offsets, pair_token, pos, pair_slot, status, nullptr, 0u, kItemRows, nullptr, 0u);
    return hipGetLastError();
}

static bool gu_lds_routed(const kq_launch_moe_dims *d, const kq_launch_moe_weights *w) {
    return kq_launch_gu_lds_supported(w->gate_type, d->hidden) != 0;
}

extern "C" void *kq_launch_moe_grouped_stage(const kq_launch_moe_dims *d,
                                             const kq_launch_moe_weights *w,
                                             const kq_launch_moe_ws *ws) {
    return gu_lds_routed(d, w) ? (void *)ws->outp : nullptr;
}

static hipError_t launch_combine(const kq_launch_moe_dims *d, const kq_launch_moe_ws *ws,
                                 uint32_t tokens, float *out, uint32_t *status, hipStream_t s) {
    hipLaunchKernelGGL(moe_combine, dim3((d->hidden / 4u + 255u) / 256u, tokens), dim3(256), 0, s,
                       ws->outp, ws->pos, ws->order, ws->weights, ws->shared_scale, tokens,
                       d->top_k, d->hidden, out, status);
    return hipGetLastError();
}

/* Whether the 64-token products (kq_gemm.hip) are the faster ones. Their items
 * are few and large: with few experts the device is not filled, and what is
 * left in a last round weighs more. Whole layer, 16-token passes / 64-token
 * products, us, at tokens per expert:
 *   2560 x 640, Q4_K / Q5_1 (Q5_K / Q8_0 within 10 % of it):
 *     512 experts  16: 808 / 861, 20: 1024 / 955, 50: 2105 / 1572
 *     256          20: 550 / 551, 24: 592 / 570, 50: 1046 / 819
 *     128          32: 402 / 416, 44: 504 / 461
 *     64           50: 304 / 328, 64: 378 / 362, 80: 452 / 432
 *     32           50: 251 / 250, 80: 314 / 316, 120: 440 / 335
 *     16           80: 231 / 240, 120: 269 / 252;   8  120: 200 / 223
 *   2048 x 512, Q4_K / Q6_K, whose mixed-tile passes keep up for longer:
 *     512 experts  32: 783 / 818, 44: 1028 / 968, 120: 2652 / 2149
 *     256          44: 509 / 512, 80: 871 / 911, 120: 1267 / 1150
 *     64           80: 235 / 271, 120: 320 / 286;   16  80: 117 / 127, 120: 137 / 130 */
static bool wide_faster(uint64_t pairs, uint32_t experts, bool mixed) {
    if (pairs >= UINT64_C(100) * experts && pairs >= 1500u) return true;
    return mixed ? pairs >= UINT64_C(44) * experts && pairs >= 22000u
                 : pairs >= UINT64_C(12) * experts + 2900u;
}

static bool wide_supported(const kq_launch_moe_dims *d, const kq_launch_moe_weights *w,
                           uint32_t tokens, bool lds_shared, bool mixed) {
    const uint32_t npos = tokens * d->top_k + tokens;
    if (!gu_lds_routed(d, w) ||
        !wide_faster((uint64_t)tokens * d->top_k, d->experts, mixed) ||
        !kq_launch_gm_gate_up_supported(w->gate_type, d->inter, d->hidden, tokens) ||
        !kq_launch_gm_matrix_supported(w->down_type, d->hidden, d->inter, npos))
        return false;
    if (lds_shared) return w->shared_down_type == w->down_type;
    return w->shared_gate_type == KQ_LAUNCH_Q8_0 && w->shared_down_type == KQ_LAUNCH_Q8_0 &&
           kq_launch_gm_matrix_supported(KQ_LAUNCH_Q8_0, d->inter, d->hidden, tokens) &&
           kq_launch_gm_matrix_supported(KQ_LAUNCH_Q8_0, d->hidden, d->inter, npos);
}

/* gate/up and down of every position into ws->outp */
static hipError_t launch_wide(const kq_launch_moe_dims *d, const kq_launch_moe_weights *w,
                              uint32_t tokens, const kq_launch_moe_ws *ws, bool lds_shared,
                              uint32_t *status, hipStream_t s) {
    const size_t tk = (size_t)tokens * d->top_k, npos = tk + tokens;
    hipError_t e = kq_launch_gm_gate_up(w->gate_type, w->gate, w->up, w->shared_gate, w->shared_up,
                                        d->inter, d->hidden, ws->outp, tokens, d->top_k,
                                        ws->perm_tok, ws->gitems, ws->act, status, s);
    if (e == hipSuccess && !lds_shared) {
        /* the Q8_0 shared expert from the same split (kq_stage.h), its
         * gate and up products in dstage, free until the down split */
        const kq::StagedX st = kq::staged_at(ws->outp, tokens, d->hidden);
        e = kq_launch_gm_dense(KQ_LAUNCH_Q8_0, w->shared_gate, w->shared_up, d->inter, d->hidden,
                               st.xh, st.xl, st.sig, tokens, (float *)ws->dstage, status, s);
        if (e == hipSuccess)
            e = kq_launch_dense_swiglu((const float *)ws->dstage, 1u, tokens, d->inter,
                                       ws->act + tk * d->inter, status, s);
    }
    _Float16 *xh = (_Float16 *)ws->dstage, *xl = xh + npos * d->inter;
    int *sig = (int *)(xl + npos * d->inter);
    if (e == hipSuccess)
        e = kq_launch_dense_split(ws->act, (uint32_t)npos, d->inter, xh, xl, sig, 0, status, s);
    if (e == hipSuccess)
        e = kq_launch_gm_down(w->down_type, w->down, w->shared_down, d->hidden, d->inter, xh, xl,
                              sig, tokens, d->top_k, ws->gitems, ws->outp, status, s);
    if (e == hipSuccess && !lds_shared)
        e = kq_launch_gm_dense(KQ_LAUNCH_Q8_0, w->shared_down, nullptr, d->hidden, d->inter,
                               xh + tk * d->inter, xl + tk * d->inter, sig + tk, tokens,
                               ws->outp + tk * d->hidden, status, s);
    return e;
}

extern "C" hipError_t kq_launch_moe_grouped(const kq_launch_moe_dims *d,
                                            const kq_launch_moe_weights *w, const float *hidden,
                                            uint32_t tokens, const kq_launch_moe_ws *ws,
                                            int staged, float *out, uint32_t *status,
                                            hipStream_t s) {
    /* Q4_K and Q5_K gate/up rows stream through LDS (kq_grouped_gu.hip) from
     * activations split once per token into the start of outp, which only
     * the down pass writes later; the work list the permutation builds for
     * it (gitems) also drives the Q6_K down pass (kq_grouped_dn.hip) */
    const bool lds_routed = gu_lds_routed(d, w);
    const bool lds_shared = lds_routed && w->shared_gate_type == w->gate_type;
    /* the mixed-tile gate/up pass (hidden 2048) records each position's
     * largest activation, and the Q6_K pair down pass (intermediate 512)
     * then splits its own operand: no dn_stage. The maxima live in dstage,
     * which only dn_stage and the dense shared expert use otherwise. */
    const bool fused_split = lds_shared && d->hidden == 2048u && d->inter == 512u &&
                             w->down_type == KQ_LAUNCH_Q6_K &&
                             w->shared_down_type == KQ_LAUNCH_Q6_K;
    /* many tokens per expert: 64 of them against each decoded weight */
    const bool wide = wide_supported(d, w, tokens, lds_shared, fused_split);
    uint32_t *posmax = fused_split && !wide ? (uint32_t *)ws->dstage : nullptr;
    hipLaunchKernelGGL(moe_permute, dim3(1), dim3(1024), 0, s, ws->ids, tokens, d->top_k,
                       d->experts, ws->offsets, ws->perm_tok, ws->pos, nullptr, status,
                       lds_routed ? (uint32_t *)ws->gitems : nullptr, lds_shared ? 1u : 0u,
                       wide ? kWideItemRows : kItemRows, posmax, posmax != nullptr ? tokens * (d->top_k + 1u) : 0u);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const uint8_t *g = (const uint8_t *)w->gate, *u = (const uint8_t *)w->up;
    const uint8_t *sg = (const uint8_t *)w->shared_gate, *su = (const uint8_t *)w->shared_up;
    const uint32_t E = d->experts;
    const uint32_t sh_wgs = (tokens + kSharedChunks * kTile - 1u) / (kSharedChunks * kTile);
    /* gate/up + SwiGLU, then down: the routed experts' workgroups and the
     * shared expert's in one launch when their formats agree */
    if (lds_routed && !staged) {
        e = kq_launch_gu_stage(hidden, tokens, d->hidden, ws->outp, status, s);
        if (e != hipSuccess) return e;
    }
    if (wide) {
        e = launch_wide(d, w, tokens, ws, lds_shared, status, s);
        if (e != hipSuccess) return e;
        return launch_combine(d, ws, tokens, out, status, s);
    }
    if (lds_routed) {
        e = kq_launch_gu_lds(w->gate_type, d->hidden, g, u, sg, su, ws->outp, ws->offsets,
                             ws->perm_tok, E, tokens, d->top_k, d->inter, lds_shared ? 1 : 0, 1,
                             ws->gitems, ws->act, posmax, status, s);
        if (e == hipSuccess && !lds_shared && w->shared_gate_type == KQ_LAUNCH_Q8_0 &&
            kq_launch_dense_q8_supported(d->inter, d->hidden, tokens)) {
            /* a Q8_0 shared expert sees every token: the dense product on
             * the same per-token split (kq_stage.h: xh [T][H], xl [T][H],
             * the 32-column sums [T][H/128][8] fp16, sig [T]), its rows
             * after the routed pairs' */
            const uint8_t *st = (const uint8_t *)ws->outp;
            const size_t th = (size_t)tokens * d->hidden;
            const int *sig =
                (const int *)(st + th * 4u + (size_t)tokens * (d->hidden / 128u) * 16u);
            float *sact = ws->act + (size_t)tokens * d->top_k * d->inter;
            /* the columns in up to four runs (more workgroups for the few
             * rows), their gate/up partials in dstage (free until the down
             * pass), summed in order with the SwiGLU */
            const uint32_t sp = kq_launch_dense_q8_splits(d->hidden, 4u);
            const uint64_t need = (uint64_t)sp * tokens * 2u * d->inter * 4u;
            const uint32_t ai = d->inter > d->shared_inter ? d->inter : d->shared_inter;
            if (sp > 1u && need <= kq_launch_dn_stage_bytes(tokens * (d->top_k + 1u), ai)) {
                e = kq_launch_dense_q8(sg, su, d->inter, d->hidden, st, st + th * 2u, sig, tokens,
                                       4u, (float *)ws->dstage, status, s);
                if (e == hipSuccess)
                    e = kq_launch_dense_swiglu((const float *)ws->dstage, sp, tokens, d->inter,
                                               sact, status, s);
            } else {
                e = kq_launch_dense_q8(sg, su, d->inter, d->hidden, st, st + th * 2u, sig, tokens,
                                       1u, sact, status, s);
            }
        } else if (e == hipSuccess && !lds_shared) {
            e = pass_any<2>(w->shared_gate_type, d->hidden, g, u, sg, su, hidden, ws->offsets,
                            ws->perm_tok, E, tokens, d->top_k, d->inter, E, sh_wgs, ws->act,
                            status, s);
        }
    } else if (w->shared_gate_type == w->gate_type) {
        e = pass_any<2>(w->gate_type, d->hidden, g, u, sg, su, hidden, ws->offsets, ws->perm_tok,
                        E, tokens, d->top_k, d->inter, 0u, E + sh_wgs, ws->act, status, s);
    } else {
        e = pass_any<2>(w->gate_type, d->hidden, g, u, sg, su, hidden, ws->offsets, ws->perm_tok,
                        E, tokens, d->top_k, d->inter, 0u, E, ws->act, status, s);
        if (e == hipSuccess)
            e = pass_any<2>(w->shared_gate_type, d->hidden, g, u, sg, su, hidden, ws->offsets,
                            ws->perm_tok, E, tokens, d->top_k, d->inter, E, sh_wgs, ws->act,
                            status, s);
    }
    if (e != hipSuccess) return e;
    const uint8_t *dn = (const uint8_t *)w->down, *sd = (const uint8_t *)w->shared_down;
    if (lds_shared && w->down_type == KQ_LAUNCH_Q6_K && w->shared_down_type == KQ_LAUNCH_Q6_K &&
        kq_launch_dn_lds_supported(d->inter)) {
        /* over the gate/up pass's item list (routed and shared chunks) */
        e = kq_launch_dn_lds(d->inter, d->hidden, dn, sd, ws->act, tokens, d->top_k, ws->gitems,
                             ws->dstage, posmax, ws->outp, status, s);
    } else if (lds_routed && kq_launch_dn_small_supported(w->down_type, d->inter) &&
               (!lds_shared || w->shared_down_type == w->down_type)) {
        /* Q5_1 or Q8_0 rows through the same per-wave LDS-DMA pipeline,
         * over the item list (the shared expert's chunks are in it when its
         * gate/up ran in the LDS gate/up pass; otherwise it runs below) */
        e = kq_launch_dn_small(w->down_type, d->inter, d->hidden, dn, sd, ws->act, tokens,
                               d->top_k, ws->gitems, ws->dstage, ws->outp, status, s);
        const size_t tk = (size_t)tokens * d->top_k;
        if (e == hipSuccess && !lds_shared && w->shared_down_type == KQ_LAUNCH_Q8_0 &&
            kq_launch_dense_q8_supported(d->hidden, d->inter, tokens)) {
            /* the dstage split above holds every position in natural order,
             * the shared expert's rows last */
            uint8_t *xs = (uint8_t *)ws->dstage;
            const size_t npos = tk + tokens, xb = npos * d->inter * 2u;
            e = kq_launch_dense_q8(sd, nullptr, d->hidden, d->inter, xs + tk * d->inter * 2u,
                                   xs + xb + tk * d->inter * 2u, (const int *)(xs + 2u * xb) + tk,
                                   tokens, 1u, ws->outp + tk * d->hidden, status, s);
        } else if (e == hipSuccess && !lds_shared) {
            e = pass_any<1>(w->shared_down_type, d->inter, dn, nullptr, sd, nullptr, ws->act,
                            ws->offsets, ws->perm_tok, E, tokens, d->top_k, d->hidden, E, sh_wgs,
                            ws->outp, status, s);
        }
    } else if (w->shared_down_type == w->down_type) {
        e = pass_any<1>(w->down_type, d->inter, dn, nullptr, sd, nullptr, ws->act, ws->offsets,
                        ws->perm_tok, E, tokens, d->top_k, d->hidden, 0u, E + sh_wgs, ws->outp,
                        status, s);
    } else {
        e = pass_any<1>(w->down_type, d->inter, dn, nullptr, sd, nullptr, ws->act, ws->offsets,
                        ws->perm_tok, E, tokens, d->top_k, d->hidden, 0u, E, ws->outp, status, s);
        const size_t tk = (size_t)tokens * d->top_k;
        if (e == hipSuccess && w->shared_down_type == KQ_LAUNCH_Q8_0 &&
            kq_launch_dense_q8_supported(d->hidden, d->inter, tokens)) {
            /* a Q8_0 shared expert's down on the dense product: its T
             * activation rows (after the routed pairs') split into dstage,
             * which only the LDS down pass uses */
            uint8_t *xs = (uint8_t *)ws->dstage;
            const size_t ti = (size_t)tokens * d->inter;
            e = kq_launch_dense_split(ws->act + tk * d->inter, tokens, d->inter, xs, xs + ti * 2u,
                                      (int *)(xs + ti * 4u), 0, status, s);
            if (e == hipSuccess)
                e = kq_launch_dense_q8(sd, nullptr, d->hidden, d->inter, xs, xs + ti * 2u,
                                       (const int *)(xs + ti * 4u), tokens, 1u,
                                       ws->outp + tk * d->hidden, status, s);
        } else if (e == hipSuccess) {
            e = pass_any<1>(w->shared_down_type, d->inter, dn, nullptr, sd, nullptr, ws->act,
                            ws->offsets, ws->perm_tok, E, tokens, d->top_k, d->hidden, E, sh_wgs,
                            ws->outp, status, s);
        }
    }
    if (e != hipSuccess) return e;
    return launch_combine(d, ws, tokens, out, status, s);
}

/* y[t] = W x[t] for every token: a Q8_0 matrix against many activation
 * rows on MFMA, as the grouped pass runs a shared matrix (16-token chunks,
 * one per workgroup), so the weights stream once per chunk instead of once
 * per four tokens */
extern "C" int kq_launch_gemm_q8_0_supported(uint32_t rows, uint32_t cols) {
    return rows != 0u && pass_dim<KQ_LAUNCH_Q8_0, 1>(cols);
}

extern "C" hipError_t kq_launch_gemm_q8_0(const void *W, uint32_t rows, uint32_t cols,
                                          const float *x, uint32_t tokens, float *y,
                                          uint32_t *status, hipStream_t s) {
    if (!kq_launch_gemm_q8_0_supported(rows, cols) || tokens == 0u) return hipErrorInvalidValue;
    const uint32_t ny = (tokens + kTile - 1u) / kTile;
    return pass_cols<KQ_LAUNCH_Q8_0, 1>(cols, nullptr, nullptr, (const uint8_t *)W, nullptr, x,
                                        nullptr, nullptr, 0u, tokens, 0u, rows, 0u, ny, 1u, y,
                                        status, s);
}
