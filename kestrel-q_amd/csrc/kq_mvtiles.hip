/*
 * kq_mvtiles.hip — y = W x on the matrix cores: GGUF Q4_K, Q5_K, Q6_K, Q8_0,
 * Q5_1 and IQ4_NL rows, 2 to 8 activation columns (and one column of widths
 * that the row engine takes in several launches).
 *
 * Restates the row loop of kq_weight_provider_linear_f32
 * (src/kq_weight_provider.c:464-475) for several activation vectors.
 *
 * The row engine (kq_rowdot.h) pays its dot per column: at four columns it
 * holds 4 x 32 activations a lane, and more than four take another launch
 * that reads the weights again. Here the weights are read and decoded once
 * for up to eight columns:
 *
 *   - One 16x16x32 fp16 step multiplies 16 weight rows by 16 operand rows,
 *     which hold the columns in parts (Rows, below): four columns in four
 *     parts each, the binary32 values exactly; eight columns in two parts
 *     (~23 bits) where the row engine rounds its columns too, or in four on
 *     two operands where it does not. The values are scaled by a power of two
 *     per column and 256-column unit.
 *   - A workgroup walks a contiguous run of 16-row tiles. A row is cut into
 *     units of 256 columns; wave w multiplies unit c nw + w of every row in
 *     the tile's c-th of NC chunks. Its activation operands, 32 registers a
 *     unit each, are built once and stay in registers for the whole run.
 *   - A chunk (16 rows x nw units) is copied into an LDS ring by 16-byte
 *     LDS-DMA loads spread over the waves, PD chunks ahead of the one being
 *     multiplied. Rows sit at an odd pitch of 16-byte units, so the 16 rows
 *     a step reads hit distinct banks.
 *   - Each wave adds its parts' product rows and leaves its columns x 16 rows
 *     in LDS; after the next barrier 16 threads a column add the waves in
 *     order, store, and keep the argmax partials: one per workgroup and
 *     column.
 *
 * A scale of 256 columns loses what lies far below the unit's largest value.
 * Columns that hold such values (least_value(), least_group()) are found while
 * the operand is built, and the workgroups then multiply the rows in binary32
 * on the vector ALU (10240 x 2560 Q8_0, 8 columns: 99 us; row engine 74).
 *
 * Codes enter fp16 exactly. Q4_K and Q5_K fold the 6-bit sub-block scale into
 * the weight, taken from the middle of the codes' range (at most 1008, exact),
 * and add the mins and the middle with two small steps against the columns'
 * sub-block sums; Q6_K takes one 16x16x16 step per 16-column sub-block, the
 * 32-weight formats one 16x16x32 step per block, scaled in fp32.
 *
 * Bound: HBM for matrices that fill the device, the first loads' latency
 * and the operand's build below that. Against the row engine: 10240 x 2560
 * Q8_0 at 8 columns 76.7 -> 12.3 us (2.3 TB/s), the 248320 x 2560 Q8_0 head
 * at 5 columns 273 -> 136 us (5.0 TB/s). Two operands keep one workgroup per
 * CU: 40000 x 2048 at 8 columns, Q5_K 23 us (row engine 53), Q5_1 37
 * (46). Error against binary64 sums of normal
 * activations 0.7-1.3e-7 of the result in every format (row engine
 * 1.7-5.7e-7).
 */
#include "kq_launch.h"
#include "kq_device.h"
#include "kq_dma.h"
#include "kq_mfma.h"

namespace {

using namespace kq::mf;

constexpr uint32_t kT = 16;      /* rows per tile */
constexpr uint32_t kCols = 8;    /* activation columns */
constexpr int kTiny = 24;        /* the last two parts carry 2^24 */
constexpr uint32_t kMaxPd = 4;   /* chunks in flight, at most */

/* eight halves as four packed registers from here on: without the asm the
 * compiler keeps the unpacked values and packs them again at every use */
__device__ __forceinline__ h8 pinned(uint32_t x, uint32_t y, uint32_t z, uint32_t w) {
    asm volatile("" : "+v"(x), "+v"(y), "+v"(z), "+v"(w));
    return __builtin_bit_cast(h8, kq_u32x4{x, y, z, w});
}
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
}
/* the value of lane l ^ 8 (a rotation by 8 within the row of 16 lanes) */
__device__ __forceinline__ uint32_t ror8(uint32_t x) { return dpp<0x128>(x); }
__device__ __forceinline__ float ror8(float x) { return __uint_as_float(ror8(__float_as_uint(x))); }
/* of lanes l ^ 1 and l ^ 2 */
__device__ __forceinline__ uint32_t quad1(uint32_t x) { return dpp<0xb1>(x); }
__device__ __forceinline__ uint32_t quad2(uint32_t x) { return dpp<0x4e>(x); }
__device__ __forceinline__ float quad1(float x) { return __uint_as_float(quad1(__float_as_uint(x))); }
__device__ __forceinline__ float quad2(float x) { return __uint_as_float(quad2(__float_as_uint(x))); }
__device__ __forceinline__ uint32_t mag(float x) { return __float_as_uint(x) & 0x7fffffffu; }

/* maximum over the four lanes (i, 0 .. 3), or over (i, g) and (i, g ^ 1) */
__device__ __forceinline__ uint32_t max16(uint32_t v) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return max((uint32_t)r[0], (uint32_t)r[1]);
}
__device__ __forceinline__ uint32_t max_groups(uint32_t v) {
    v = max16(v);
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return max((uint32_t)r[0], (uint32_t)r[1]);
}

/* Two binary32 values (at most 2^15) as N halves each, v = p0 + p1 + 2^-24 (p2 +
 * p3). N = 4: exact where |v| is 0 or at least 2^-25, whose last bit is 2^-48;
 * below that the error is at most 2^-49. N = 2: to 2^-23 |v| or 2^-25, the
 * larger. (The differences are exact.) */
template <int N>
__device__ __forceinline__ void split(float a, float b, h2 (&p)[N]) {
    typedef float f2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int n = 0; n < N; ++n) {
        p[n] = __builtin_convertvector((f2{a, b}), h2);
        a = fmaf((float)p[n].x, -1.0f, a);
        b = fmaf((float)p[n].y, -1.0f, b);
        if (n == 1) {
            a *= 0x1p24f;
            b *= 0x1p24f;
        }
    }
}

/* How the 16 operand rows hold the columns.
 *   kQuad: 4 columns, rows 4c .. 4c + 3 the parts of column c.
 *   kEight: 8 columns on two operands: rows 0 .. 7 parts 0 (first operand) and
 *     1 (second), rows 8 .. 15 parts 2 and 3.
 *   kPair: 8 columns, rows 0 .. 7 part 0, rows 8 .. 15 part 1, nothing more.
 * The row engine multiplies Q4_K, Q6_K and Q8_0 with 23-bit integers in a
 * scale per 16 columns, the other formats with the binary32 values; more than
 * four columns of the former take kPair, of the latter kEight. */
enum Rows : uint32_t { kQuad, kPair, kEight };
constexpr bool is_binary32(uint32_t f) {
    return f == KQ_LAUNCH_Q5_K || f == KQ_LAUNCH_Q5_1 || f == KQ_LAUNCH_IQ4_NL;
}
constexpr uint32_t columns_of(Rows m) { return m == kQuad ? 4u : 8u; }
constexpr uint32_t operands_of(Rows m) { return m == kEight ? 2u : 1u; }

/* What the operands take, in the scaled values (largest in [2^14, 2^15)). Four
 * parts hold a value as binary32 does down to least_value() (asked of the
 * formats that the row engine multiplies so). 16 columns are held as a scale of
 * their own holds them if one reaches least_group(): two parts are off by 2^-25,
 * four by 2^-49, the scale by 2^-23 of their largest; and the sums of such
 * columns, which are scaled down again, if one does. Anything smaller but zeros
 * goes to the binary32 rows. (Asked of single values, the 320 SiLU outputs of a
 * saturated rank projection went there in most calls: 20 us more on the 68 of a
 * one-token block.) */
template <uint32_t FMT, Rows M>
constexpr float least_value() {
    return M == kQuad && !is_binary32(FMT) ? 0.0f : 0x1p-25f; /* kPair: not looked at */
}
template <uint32_t FMT, Rows M>
constexpr float least_group() {
    return M == kPair ? 0x1p-2f : is_k(FMT) ? 0x1p-20f : FMT == KQ_LAUNCH_Q5_1 ? 0x1p-16f
                      : is_binary32(FMT) ? 0.0f : 0x1p-25f;
}

/* The column of its unit that lane k-group g's element e of operand step s
 * stands for. A step's k order is free as long as both operands agree; it
 * follows the bytes a lane reads in one piece. Q6_K: elements 0..3 and 4..7
 * are the 16x16x16 steps 2s and 2s + 1, step i = 8 n + 4 h + q being
 * sub-block 8 n + 2 q + h. */
template <uint32_t FMT>
__device__ __forceinline__ uint32_t column_of(uint32_t g, uint32_t s, uint32_t e) {
    if constexpr (is_k(FMT)) return 64u * g + 8u * s + e;
    if constexpr (FMT == KQ_LAUNCH_Q6_K) {
        const uint32_t i = 2u * s + (e >> 2), n = i >> 3, h = (i >> 2) & 1u, q = i & 3u;
        return 128u * n + 32u * q + 16u * h + 4u * g + (e & 3u);
    }
    return 32u * s + 8u * g + e;
}

/* what a unit's min term needs of the columns: their sub-block sums times
 * 2^-5, sums 4g .. 4g + 3 on k-groups 0 and 1 (Q4_K, Q5_K; kPair: their parts
 * 2 and 3 times 2^-13 on k-groups 2 and 3, against mins times 2^-11); their block sums
 * times 2^-9 on k-groups 0 and 1 (against m) and times 16 2^-9 on 2 and 3
 * (against d, for the codes' middle 16) (Q5_1) */
constexpr bool has_min(uint32_t f) { return is_k(f) || f == KQ_LAUNCH_Q5_1; }

/* IQ4_NL: the values of four nibbles (src/kq_numeric.c) plus 128 */
__device__ __forceinline__ uint32_t iq4_codes(uint32_t n) {
    const uint32_t lo = __builtin_amdgcn_perm(0x766a5d4fu, 0x3f2d1801u, n & 0x07070707u);
    const uint32_t hi = __builtin_amdgcn_perm(0xf1d9c5b5u, 0xa6998d81u, n & 0x07070707u);
    const uint32_t b3 = (n >> 3) & 0x01010101u, m = (b3 << 8) - b3;
    return (hi & m) | (lo & ~m);
}

/* One unit of row j of the tile times the activation operands: returns
 * lane (j, g)'s products of operand rows 4g .. 4g + 3, summed over the G
 * operands, in the operand's scale. p: the unit's first byte in LDS (p - off is 4-byte aligned, off 0
 * or 2); live: steps that hold columns (8 but for
 * a row's last unit); real: row j exists. */
template <uint32_t FMT, Rows M, uint32_t G>
__device__ __forceinline__ f4 unit_product(const uint8_t *p, uint32_t off, uint32_t g,
                                           uint32_t live, bool real, const h8 (&A)[G][8],
                                           const h4 (&sums)[G], bool &malformed) {
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
    /* the operands' products apart: chained, Q5_1 errs by a tenth more */
    auto step = [&](uint32_t s, h8 b) {
        f4 t = mfma32(A[0][s], b, zero);
        if constexpr (G == 2u) t += mfma32(A[1][s], b, zero);
        return t;
    };
    auto min_step = [&](h4 b) {
        f4 t = mfma16(sums[0], b, zero);
        if constexpr (G == 2u) t += mfma16(sums[1], b, zero);
        return t;
    };
    f4 acc = zero;
    static_assert(G == 1u || is_binary32(FMT), "two operands hold binary32 values");
    if constexpr (is_k(FMT)) {
        constexpr bool Q5 = FMT == KQ_LAUNCH_Q5_K;
        constexpr uint32_t QS = Q5 ? 48u : 16u;
        const uint4 hd = *(const uint4 *)p;
        const uint4 qa = *(const uint4 *)(p + QS + 32u * g);
        const uint4 qb = *(const uint4 *)(p + QS + 16u + 32u * g);
        uint4 ha = {0u, 0u, 0u, 0u}, hb = {0u, 0u, 0u, 0u};
        if constexpr (Q5) {
            ha = *(const uint4 *)(p + 16u);
            hb = *(const uint4 *)(p + 32u);
        }
        const float d = half_bits(hd.x), dmin = half_bits(hd.x >> 16);
        malformed |= real && (!kq_isfinite(d) || !kq_isfinite(dmin));
        constexpr float kMid = k_mid(FMT);
        /* k-group g: sub-blocks 2g (steps 0..3) and 2g + 1 (steps 4..7) */
        const KPair<FMT, true> sc(hd, g);
        f4 t[G];
#pragma unroll
        for (uint32_t o = 0; o < G; ++o) t[o] = zero;
#pragma unroll
        for (uint32_t s = 0; s < 8u; ++s) {
            const h8 b = sc.weights(s >> 2, g, dword_of(qa, qb, s & 3u, 0u), dword_of(qa, qb, s & 3u, 1u),
                                    dword_of(ha, hb, s & 3u, 0u), dword_of(ha, hb, s & 3u, 1u));
#pragma unroll
            for (uint32_t o = 0; o < G; ++o) t[o] = mfma32(A[o][s], b, t[o]);
        }
        acc = t[0];
        if constexpr (G == 2u) acc += t[1];
        auto halves = [&](uint32_t b) {
            if constexpr (M == kPair) {
                const _Float16 f = g < 2u ? (_Float16)1.0f : (_Float16)0x1p-11f;
                return byte_halves(b) * h4{f, f, f, f};
            } else {
                return byte_halves(g < 2u ? b : 0u);
            }
        };
        const f4 mm = min_step(halves(k_mins(hd, g & 1u)));
        const f4 ss = min_step(halves(k_centres(hd, g & 1u)));
        /* the sums carry 2^-5 */
        const float dw = d * 0x1p14f, dc = d * (kMid * 32.0f), dm = dmin * 32.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[k] = fmaf(dw, acc[k], fmaf(dc, ss[k], -dm * mm[k]));
        return acc;
    } else if constexpr (FMT == KQ_LAUNCH_Q6_K) {
        const h2 bias = splat(-1056.0f); /* 1024 + 32 */
        const uint32_t *w = (const uint32_t *)(p - off);
        auto win = [&](uint32_t o) { return kq_align2(w[o / 4u + 1u], w[o / 4u], off); };
        const float d = half_bits(off ? w[52] >> 16 : w[52]); /* bytes 208, 209 */
        malformed |= real && !kq_isfinite(d);
#pragma unroll
        for (uint32_t n = 0; n < 2u; ++n) {
            const uint32_t sc[2] = {win(192u + 8u * n), win(196u + 8u * n)};
#pragma unroll
            for (uint32_t h = 0; h < 2u; ++h) {
                /* w indexed per lane by g: byte offsets 4g more */
                const uint32_t *wg = w + g;
                auto wing = [&](uint32_t o) { return kq_align2(wg[o / 4u + 1u], wg[o / 4u], off); };
                const uint32_t a = wing(64u * n + 16u * h), b = wing(64u * n + 16u * h + 32u);
                const uint32_t q = wing(128u + 32u * n + 16u * h);
                const uint32_t c[4] = {(a & 0x0f0f0f0fu) | ((q << 4) & 0x30303030u),
                                       (b & 0x0f0f0f0fu) | ((q << 2) & 0x30303030u),
                                       ((a >> 4) & 0x0f0f0f0fu) | (q & 0x30303030u),
                                       ((b >> 4) & 0x0f0f0f0fu) | ((q >> 2) & 0x30303030u)};
#pragma unroll
                for (uint32_t k = 0; k < 4u; ++k) {
                    const uint32_t i = 8u * n + 4u * h + k;
                    const h2 w0 = bytes_lo(c[k]) + bias, w1 = bytes_hi(c[k]) + bias;
                    const h8 &as = A[0][i >> 1];
                    const h4 a4 = (i & 1u) ? h4{as[4], as[5], as[6], as[7]}
                                           : h4{as[0], as[1], as[2], as[3]};
                    const f4 t = mfma16(a4, h4{w0.x, w0.y, w1.x, w1.y}, zero);
                    const uint32_t sub = 2u * k + h; /* of this half's eight */
                    const int8_t s8 = (int8_t)((sc[sub >> 2] >> (8u * (sub & 3u))) & 0xffu);
                    const float ds = d * (float)s8;
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[r] = fmaf(ds, t[r], acc[r]);
                }
            }
        }
        return acc;
    } else {
        const uint32_t *w = (const uint32_t *)p;
        uint32_t mins[4] = {0u, 0u, 0u, 0u};
        const uint32_t shn = g >= 2u ? 4u : 0u; /* Q5_1, IQ4_NL: this lane's nibbles */
        /* Q5_1 codes enter as q - 16 and 16 d joins the min; as q where there is
         * none, whose zero codes are zero weights */
        h2 bias = splat(FMT == KQ_LAUNCH_Q5_1 ? -1040.0f : -1152.0f);
#pragma unroll
        for (uint32_t s = 0; s < 8u; ++s) {
            uint32_t c0, c1;
            float d;
            if constexpr (FMT == KQ_LAUNCH_Q8_0) {
                /* block s at byte 34 s: codes of k-group g at 34 s + 2 + 8 g,
                 * offset by 128 into unsigned bytes */
                if (s % 2u == 0u) {
                    const uint32_t *b = w + 17u * (s / 2u);
                    d = half_bits(b[0]);
                    const uint32_t q0 = b[2u * g], q1 = b[2u * g + 1u], q2 = b[2u * g + 2u];
                    c0 = kq_align2(q1, q0, 2u) ^ 0x80808080u;
                    c1 = kq_align2(q2, q1, 2u) ^ 0x80808080u;
                } else {
                    const uint32_t *b = w + (34u * s - 2u) / 4u;
                    d = half_bits(b[0] >> 16);
                    c0 = b[1u + 2u * g] ^ 0x80808080u;
                    c1 = b[2u + 2u * g] ^ 0x80808080u;
                }
                malformed |= real && s < live && !kq_isfinite(d);
            } else if constexpr (FMT == KQ_LAUNCH_Q5_1) {
                const uint32_t *b = w + 6u * s;
                const uint32_t dm = b[0], hb = (b[1] >> (8u * g)) & 0xffu;
                const uint32_t *q = b + 2u + 2u * (g & 1u);
                c0 = ((q[0] >> shn) & 0x0f0f0f0fu) | spread4(hb & 15u);
                c1 = ((q[1] >> shn) & 0x0f0f0f0fu) | spread4(hb >> 4);
                d = half_bits(dm);
                malformed |= real && s < live && (!kq_isfinite(d) || !kq_isfinite(half_bits(dm >> 16)));
                /* min term: m of blocks 4g .. 4g + 3 (g < 2), then d of
                 * blocks 4 (g - 2) .. */
                const bool zero_min = (dm & 0x7fff0000u) == 0u;
                bias = splat(zero_min ? -1024.0f : -1040.0f);
                if (s < live)
                    mins[s & 3u] = (s >> 2) == (g & 1u) ? (g < 2u ? dm >> 16 : zero_min ? 0u : dm & 0xffffu)
                                                        : mins[s & 3u];
            } else {
                /* block s at byte 18 s: this lane's eight nibbles at
                 * 18 s + 2 + 8 (g & 1) */
                uint32_t q0, q1;
                if (s % 2u == 0u) {
                    const uint32_t *b = w + 9u * (s / 2u) + 2u * (g & 1u);
                    d = half_bits(w[9u * (s / 2u)]);
                    q0 = kq_align2(b[1], b[0], 2u);
                    q1 = kq_align2(b[2], b[1], 2u);
                } else {
                    const uint32_t *b = w + (18u * s - 2u) / 4u;
                    d = half_bits(b[0] >> 16);
                    q0 = b[1u + 2u * (g & 1u)];
                    q1 = b[2u + 2u * (g & 1u)];
                }
                malformed |= real && s < live && !kq_isfinite(d);
                c0 = iq4_codes((q0 >> shn) & 0x0f0f0f0fu);
                c1 = iq4_codes((q1 >> shn) & 0x0f0f0f0fu);
            }
            if (s >= live) d = 0.0f;
            const f4 t = step(s, cat(bytes_lo(c0) + bias, bytes_hi(c0) + bias, bytes_lo(c1) + bias,
                                     bytes_hi(c1) + bias));
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[k] = fmaf(d, t[k], acc[k]);
        }
        if constexpr (FMT == KQ_LAUNCH_Q5_1) {
            const h4 bm = __builtin_bit_cast(
                h4, make_uint2((mins[0] & 0xffffu) | (mins[1] << 16), (mins[2] & 0xffffu) | (mins[3] << 16)));
            const f4 mm = min_step(bm);
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[k] = fmaf(0x1p9f, mm[k], acc[k]);
        }
        return acc;
    }
}

/* the decoded weights of columns c .. c + 3 of a row (c a multiple of 4), as
 * the CPU decodes them (src/kq_numeric.c) */
template <uint32_t FMT>
__device__ __forceinline__ void weights_at(const uint8_t *row, uint32_t c, float (&w)[4], bool &malformed) {
    auto half = [&](const uint8_t *p) {
        const float v = half_bits((uint32_t)p[0] | ((uint32_t)p[1] << 8));
        malformed |= !kq_isfinite(v);
        return v;
    };
    auto dword = [](const uint8_t *p) {
        uint32_t v;
        __builtin_memcpy(&v, p, 4);
        return v;
    };
    constexpr uint32_t BC = block_cols(FMT);
    const uint8_t *b = row + c / BC * (unit_bytes(FMT) / (kUnit / BC));
    const uint32_t i = c % BC, sub = i >> 5, l = i & 31u;
    uint32_t q; /* four codes */
    float d, m = 0.0f, zero = 0.0f;
    if constexpr (is_k(FMT)) {
        const uint8_t *s = b + 4u;
        const uint32_t sc = sub < 4u ? s[sub] & 63u : (s[sub + 4u] & 15u) | (s[sub - 4u] >> 6 << 4);
        const uint32_t mn = sub < 4u ? s[sub + 4u] & 63u : (s[sub + 4u] >> 4) | (s[sub] >> 6 << 4);
        q = (dword(b + (FMT == KQ_LAUNCH_Q5_K ? 48u : 16u) + 32u * (sub >> 1) + l) >> (4u * (sub & 1u))) &
            0x0f0f0f0fu;
        if constexpr (FMT == KQ_LAUNCH_Q5_K) q |= ((dword(b + 16u + l) >> sub) & 0x01010101u) << 4;
        d = half(b) * (float)sc;
        m = -(half(b + 2) * (float)mn);
    } else if constexpr (FMT == KQ_LAUNCH_Q6_K) {
        const uint32_t n = i >> 7, k = sub & 3u;
        q = ((dword(b + 64u * n + 32u * (k & 1u) + l) >> (2u * (k & 2u))) & 0x0f0f0f0fu) |
            (((dword(b + 128u + 32u * n + l) >> (2u * k)) & 0x03030303u) << 4);
        zero = 32.0f;
        d = half(b + 208) * (float)(int8_t)b[192u + 8u * n + 2u * k + (l >> 4)];
    } else if constexpr (FMT == KQ_LAUNCH_Q8_0) {
        q = dword(b + 2u + l) ^ 0x80808080u;
        zero = 128.0f;
        d = half(b);
    } else {
        const uint32_t nib = (dword(b + (FMT == KQ_LAUNCH_Q5_1 ? 8u : 2u) + (l & 15u)) >> (l >= 16u ? 4u : 0u)) &
                             0x0f0f0f0fu;
        d = half(b);
        if constexpr (FMT == KQ_LAUNCH_Q5_1) {
            q = nib | spread4((dword(b + 4u) >> l) & 15u);
            m = half(b + 2);
        } else {
            q = iq4_codes(nib);
            zero = 128.0f;
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = d * ((float)((q >> (8 * e)) & 0xffu) - zero) + m;
}

/* larger value wins, equal values keep the lower row */
__device__ __forceinline__ void argmax_merge(float &bv, uint32_t &bi, float v, uint32_t i) {
    if (v > bv || (v == bv && i < bi)) {
        bv = v;
        bi = i;
    }
}

struct MvtArgs {
    const uint8_t *W;
    uint32_t rows, cols, row_bytes, w_bytes; /* w_bytes: whole dwords */
    const float *x;
    uint32_t batch;
    float *y;
    uint32_t *status;
    float *part_v;
    uint32_t *part_i;
    uint32_t part_stride;
    uint32_t pitch, slot, pd; /* LDS: 16-byte units per row, bytes per chunk slot; slots - 1 */
    uint32_t tiles, more;     /* tiles = grid size * tiles + more */
};

/* The kernel's arguments, loaded where they are used: what only the rare or last
 * parts of the kernel read stays out of the scalar registers before them (21
 * of those were spilled otherwise, some in the loop). */
__device__ __forceinline__ const MvtArgs *late_args() {
    auto p = (const __attribute__((address_space(4))) MvtArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return (const MvtArgs *)p;
}

/* LDS-DMA instructions per wave and chunk: a chunk's 16 rows take at most
 * nw unit_bytes / 16 + 2 units each, 64 units an instruction, nw waves */
template <uint32_t FMT>
constexpr uint32_t ipw() {
    return (unit_bytes(FMT) + 32u + 63u) / 64u;
}

/* Register budget: 10 waves of up to 168 registers while a wave holds at most
 * two operands of 32, 8 of up to 256 above. */
constexpr uint32_t kNarrow = 2u;
template <uint32_t NC, Rows M>
constexpr int max_threads() {
    return NC * operands_of(M) <= kNarrow ? 640 : 512;
}

/* PART: the row's last unit holds fewer than 256 columns */
template <uint32_t FMT, uint32_t NC, bool PART, Rows M>
__global__ __launch_bounds__((max_threads<NC, M>())) void mv_tiles(MvtArgs a) {
    constexpr uint32_t KC = columns_of(M), G = operands_of(M);
    constexpr uint32_t UB = unit_bytes(FMT), IPW = ipw<FMT>();
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t nw = blockDim.x >> 6;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 15u, g = lane >> 4;
    /* ring, landing place of the padding loads, partial sums by tile parity
     * [2][nw][KC][16], the units' powers of two [NC][nw][KC], which waves hold
     * values out of the operand's reach */
    uint8_t *ring = lds, *trash = ring + (a.pd + 1u) * a.slot;
    float *part = (float *)(trash + 1024u);
    int *sigs = (int *)(part + 2u * nw * (KC * 16u));
    uint32_t *deeps = (uint32_t *)(sigs + NC * nw * KC);

    /* the first `more` workgroups walk one tile more than the others */
    const uint32_t lo = a.tiles * blockIdx.x + min(blockIdx.x, a.more);
    const uint32_t hi = lo + a.tiles + (blockIdx.x < a.more ? 1u : 0u);
    const uint32_t n_ent = (hi - lo) * NC;
    const kq_i4v wr = dma_rsrc(a.W, a.w_bytes);
    const uint32_t nu = (a.cols + kUnit - 1u) / kUnit;

    /* this wave's instructions n = w + nw q of a chunk: the lane's byte
     * offset from the chunk's first row. Tiles and chunks start on dwords;
     * a Q6_K row that does not is copied from the dword it starts in. */
    uint32_t rel[IPW];
#pragma unroll
    for (uint32_t q = 0; q < IPW; ++q) {
        const uint32_t u = (w + nw * q) * 64u + lane;
        const uint32_t r = u / a.pitch, c = u - r * a.pitch;
        rel[q] = r < kT ? ((r * a.row_bytes) & ~3u) + 16u * c : 0u;
    }
    const uint32_t n_ins = (kT * a.pitch + 63u) / 64u;
    uint32_t iss_off = lo * kT * a.row_bytes, iss_c = 0u, iss_slot = 0u;
    auto issue = [&]() {
        const uint32_t dst = lds_addr(ring) + iss_slot * a.slot;
#pragma unroll
        for (uint32_t q = 0; q < IPW; ++q) {
            const uint32_t n = w + nw * q; /* wave-uniform */
            dma16(wr, iss_off + iss_c * nw * UB + rel[q],
                  n < n_ins ? dst + 1024u * n : lds_addr(trash));
        }
        iss_slot = iss_slot == a.pd ? 0u : iss_slot + 1u;
        if (++iss_c == NC) {
            iss_c = 0u;
            iss_off += kT * a.row_bytes;
        }
    };
    /* the first chunk now, the others once the operand's activations have
     * arrived: loads return in order, and behind a full ring the activations
     * would wait for it */
    issue();

    /* the activation operands of this wave's units: lane (i, g) holds operand
     * row i of k-group g. The lanes that hold parts of one column (kQuad: four
     * neighbours; else lanes i and i + 8) divide its values between them and
     * trade their parts, so each value is scaled and split once (768 -> 350
     * VALU instructions a unit of kPair, which the smallest products feel).
     * kQuad: steps 2 q and 2 q + 1 on lane q of the four; else elements 4 q ..
     * 4 q + 3 of every step on lane i + 8 q. */
    h8 A[NC][G][8];
    h4 sums[NC][G];
    bool bad = false, deep = false;
    {
        constexpr uint32_t NV = M == kQuad ? 4u : 8u; /* float4 a lane loads and splits */
        constexpr int NP = M == kPair ? 2 : 4;        /* parts */
        const uint32_t i = lane & 15u;
        const uint32_t col = M == kQuad ? i >> 2 : i & 7u, q = M == kQuad ? i & 3u : i >> 3;
        const bool q0 = (q & 1u) != 0u, q1 = (q & 2u) != 0u;
        /* columns past the row, and columns past the batch, read as zeros */
        const KqBuf bx = kq_buf(a.x, a.batch * a.cols * 4u);
        auto load = [&](uint32_t c, uint4 (&v)[NV]) {
            const uint32_t u = c * nw + w, xo = (col * a.cols + kUnit * u) * 4u;
            const uint32_t left = u < nu && col < a.batch ? a.cols - kUnit * u : 0u;
#pragma unroll
            for (uint32_t k = 0; k < NV; ++k) {
                const uint32_t at = M == kQuad ? column_of<FMT>(g, 2u * q + (k >> 1), 4u * (k & 1u))
                                    : q0       ? column_of<FMT>(g, k, 4u)
                                               : column_of<FMT>(g, k, 0u);
                v[k] = kq_ld128(bx, at < left ? xo + 4u * at : 0x80000000u, 0u);
            }
        };
        uint4 vn[NV];
        load(0u, vn);
#pragma unroll
        for (uint32_t c = 0; c < NC; ++c) {
            float4 v[NV];
#pragma unroll
            for (uint32_t k = 0; k < NV; ++k) v[k] = __builtin_bit_cast(float4, vn[k]);
            if (c + 1u < NC) load(c + 1u, vn);
            /* largest magnitude, and less one the smallest but zero of the
             * values and of the groups' largest, as bits */
            uint32_t m = 0u, value1 = 0xffffffffu, group1 = 0xffffffffu, gm[NV];
#pragma unroll
            for (uint32_t k = 0; k < NV; ++k) {
                const uint32_t mx = mag(v[k].x), my = mag(v[k].y), mz = mag(v[k].z), mw = mag(v[k].w);
                gm[k] = max(max(mx, my), max(mz, mw));
                if constexpr (M != kPair && least_value<FMT, M>() != 0.0f) {
                    value1 = min(min(value1, mx - 1u), my - 1u);
                    value1 = min(min(value1, mz - 1u), mw - 1u);
                }
            }
            if constexpr (least_group<FMT, M>() != 0.0f) {
                /* a group. kQuad: 16 columns, a lane's (K formats), four
                 * elements of each k-group (Q6_K) or half a step of k-groups g
                 * and g ^ 1; else 8 of them, half a step or, Q6_K, four elements
                 * of two k-groups (the other 8 beside them cost registers that
                 * the widest rows do not have) */
                constexpr uint32_t N = FMT == KQ_LAUNCH_Q6_K ? 1u : is_k(FMT) ? 4u : 2u;
#pragma unroll
                for (uint32_t k = 0; k < NV; ++k) {
                    if constexpr (M == kQuad) {
                        if (k % N != 0u) continue;
                        uint32_t gk = gm[k];
#pragma unroll
                        for (uint32_t n = 1; n < N; ++n) gk = max(gk, gm[k + n]);
                        if constexpr (FMT == KQ_LAUNCH_Q6_K) gk = max_groups(gk);
                        else if constexpr (!is_k(FMT)) gk = max16(gk);
                        group1 = min(group1, gk - 1u);
                    } else {
                        gm[k] = FMT == KQ_LAUNCH_Q6_K ? max16(gm[k]) : max(gm[k], ror8(gm[k]));
                        group1 = min(group1, gm[k] - 1u);
                    }
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < NV; ++k) m = max(m, gm[k]);
            m = max(m, M == kQuad ? quad1(m) : ror8(m));
            if constexpr (M == kQuad) m = max(m, quad2(m));
            m = max_groups(m);
            /* largest magnitude into [2^14, 2^15); a column with a
             * non-finite value contributes zeros (the call fails) */
            const bool nf = m >= 0x7f800000u;
            bad |= nf;
            const int sig = !nf && m != 0u ? 15 - __builtin_amdgcn_frexp_expf(__uint_as_float(m)) : 0;
            auto below = [&](float scaled) { return max(mag(ldexpf(scaled, -sig)), 1u) - 1u; };
            deep |= !nf && (value1 < below(least_value<FMT, M>()) || group1 < below(least_group<FMT, M>()));
            if (g == 0u && (M == kQuad ? q == 0u : i < KC)) sigs[(c * nw + w) * KC + col] = sig;
            float run[2] = {0.0f, 0.0f}, by_step[NV]; /* sums over this lane's values */
            uint32_t own[4][4]; /* kQuad: a step's [part][dword] */
#pragma unroll
            for (uint32_t k = 0; k < NV; ++k) {
                if (nf) v[k] = float4{0.f, 0.f, 0.f, 0.f};
                const float xs[4] = {ldexpf(v[k].x, sig), ldexpf(v[k].y, sig), ldexpf(v[k].z, sig),
                                     ldexpf(v[k].w, sig)};
                h2 pa[NP], pb[NP];
                split<NP>(xs[0], xs[1], pa);
                split<NP>(xs[2], xs[3], pb);
                auto lo_of = [&](int n) { return __builtin_bit_cast(uint32_t, pa[n]); };
                auto hi_of = [&](int n) { return __builtin_bit_cast(uint32_t, pb[n]); };
                const float s4 = (xs[0] + xs[1]) + (xs[2] + xs[3]);
                if constexpr (M == kQuad) {
                    run[k >> 1] += s4;
#pragma unroll
                    for (int n = 0; n < NP; ++n) {
                        own[n][2u * (k & 1u)] = lo_of(n);
                        own[n][2u * (k & 1u) + 1u] = hi_of(n);
                    }
                    if ((k & 1u) == 0u) continue;
                    /* four lanes' parts of a step each to each lane's part of four steps */
                    uint32_t f[4][4]; /* [lane][dword] */
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        uint32_t l[2][2];
#pragma unroll
                        for (uint32_t n = 0; n < 2u; ++n) {
                            const uint32_t even = own[2u * n][d], odd = own[2u * n + 1u][d];
                            const uint32_t r = quad1(q0 ? even : odd);
                            l[n][0] = q0 ? r : even;
                            l[n][1] = q0 ? odd : r;
                        }
#pragma unroll
                        for (uint32_t b = 0; b < 2u; ++b) {
                            const uint32_t r = quad2(q1 ? l[0][b] : l[1][b]);
                            f[b][d] = q1 ? r : l[0][b];
                            f[2u + b][d] = q1 ? l[1][b] : r;
                        }
                    }
#pragma unroll
                    for (uint32_t b = 0; b < 4u; ++b)
                        A[c][0][2u * b + (k >> 1)] = pinned(f[b][0], f[b][1], f[b][2], f[b][3]);
                } else {
                    /* operand o: part o on rows 0 .. 7, part G + o on 8 .. 15 */
#pragma unroll
                    for (uint32_t o = 0; o < G; ++o) {
                        const uint32_t mx = lo_of(o), my = hi_of(o), tx = lo_of(G + o), ty = hi_of(G + o);
                        const uint32_t r0 = ror8(q0 ? mx : tx), r1 = ror8(q0 ? my : ty);
                        A[c][o][k] = pinned(q0 ? r0 : mx, q0 ? r1 : my, q0 ? tx : r0, q0 ? ty : r1);
                    }
                    if constexpr (has_min(FMT)) {
                        run[k >> 2] += s4;
                        by_step[k] = s4;
                    }
                }
            }
            float sm[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (is_k(FMT)) {
                /* each lane of k-group g: sub-blocks 2g and 2g + 1 */
                if constexpr (M == kQuad) {
                    float half = run[0] + run[1];
                    half += quad1(half);
                    const float other = quad2(half);
                    run[0] = q1 ? other : half;
                    run[1] = q1 ? half : other;
                } else {
                    run[0] += ror8(run[0]);
                    run[1] += ror8(run[1]);
                }
                const int src = (int)(i + 32u * (g & 1u));
                sm[0] = __shfl(run[0], src, KQ_WAVE);
                sm[1] = __shfl(run[1], src, KQ_WAVE);
                sm[2] = __shfl(run[0], src + 16, KQ_WAVE);
                sm[3] = __shfl(run[1], src + 16, KQ_WAVE);
            } else if constexpr (FMT == KQ_LAUNCH_Q5_1) {
                auto over_groups = [](float b) {
                    b += __shfl_xor(b, 16, KQ_WAVE);
                    return b + __shfl_xor(b, 32, KQ_WAVE);
                };
                if constexpr (M == kQuad) {
                    /* blocks 2 q and 2 q + 1, from lane q of the four */
                    const uint32_t b0 = __float_as_uint(over_groups(run[0]));
                    const uint32_t b1 = __float_as_uint(over_groups(run[1]));
                    const bool up = (g & 1u) != 0u;
                    sm[0] = __uint_as_float(up ? dpp<0xaa>(b0) : dpp<0x00>(b0));
                    sm[1] = __uint_as_float(up ? dpp<0xaa>(b1) : dpp<0x00>(b1));
                    sm[2] = __uint_as_float(up ? dpp<0xff>(b0) : dpp<0x55>(b0));
                    sm[3] = __uint_as_float(up ? dpp<0xff>(b1) : dpp<0x55>(b1));
                } else {
#pragma unroll
                    for (uint32_t e = 0; e < 4u; ++e) {
                        const float b0 = over_groups(by_step[e] + ror8(by_step[e]));
                        const float b1 = over_groups(by_step[e + 4u] + ror8(by_step[e + 4u]));
                        sm[e] = (g & 1u) != 0u ? b1 : b0;
                    }
                }
            }
#pragma unroll
            for (uint32_t o = 0; o < G; ++o) sums[c][o] = h4{};
            if constexpr (has_min(FMT)) {
                const float scale = FMT == KQ_LAUNCH_Q5_1 ? (g < 2u ? 0x1p-9f : 0x1p-5f)
                                    : M == kPair || g < 2u ? 0x1p-5f : 0.0f;
#pragma unroll
                for (uint32_t e = 0; e < 4u; e += 2u) {
                    h2 p[4];
                    split<4>(sm[e] * scale, sm[e + 1u] * scale, p);
#pragma unroll
                    for (uint32_t o = 0; o < G; ++o) {
                        const h2 p0 = p[0], p1 = p[1], p2 = p[2], p3 = p[3];
                        h2 r;
                        if constexpr (M == kQuad) {
                            const h2 even = q1 ? p2 : p0, odd = q1 ? p3 : p1;
                            r = q0 ? odd : even;
                        } else if constexpr (M == kEight) {
                            const h2 big = o == 0u ? p0 : p1, tiny = o == 0u ? p2 : p3;
                            r = q0 ? tiny : big;
                        } else {
                            const h2 a2 = p2 * splat(0x1p-13f), a3 = p3 * splat(0x1p-13f);
                            r = q0 ? (g < 2u ? p1 : a3) : (g < 2u ? p0 : a2);
                        }
                        sums[c][o][e] = r.x;
                        sums[c][o][e + 1u] = r.y;
                    }
                }
            }
            /* one unit's values, and the next one's on their way */
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    {
        const uint64_t any = __ballot(deep);
        if (lane == 0u) deeps[w] = (uint32_t)(any != 0ull);
    }
    for (uint32_t t = 1; t < a.pd && t < n_ent; ++t) issue();

    const uint32_t t = threadIdx.x; /* < 16 KC: output column t / 16, row t % 16 */
    float best_v = -__builtin_inff();
    uint32_t best_i = 0xffffffffu;
    bool malformed = false, nonfinite = false;
    f4 acc = {0.f, 0.f, 0.f, 0.f};
    uint32_t slot = 0u, ent = 0u;
    auto finish = [&](uint32_t tile, uint32_t parts) {
        if (t < KC * 16u) {
            const float *pp = part + (tile & 1u) * nw * (KC * 16u) + t;
            float s = 0.0f;
            for (uint32_t q = 0; q < parts; ++q) s += pp[q * (KC * 16u)];
            const uint32_t row = tile * kT + (t & 15u), col = t >> 4;
            if (row < a.rows && col < a.batch) {
                nonfinite |= !kq_isfinite(s);
                a.y[(size_t)col * a.rows + row] = s;
                argmax_merge(best_v, best_i, s, row);
            }
        }
    };
    /* the first chunk's loads have landed (those of the chunks requested after
     * it may be in flight): in this wave, then in all */
    wait_after<IPW, kMaxPd - 1u>(n_ent - 1u < a.pd - 1u ? n_ent - 1u : a.pd - 1u);
    kq_lds_barrier();
    if (__builtin_expect(__ballot(lane < nw && deeps[lane < nw ? lane : 0u] != 0u) != 0ull, 0)) {
        /* some value lies too far below its unit's largest for the operand:
         * the rows in binary32, a wave a row (every workgroup sees the same
         * values and comes here) */
        const MvtArgs *b = late_args();
        for (uint32_t tile = lo; tile < hi; ++tile) {
            for (uint32_t r = w; r < kT; r += nw) {
                const uint32_t row = tile * kT + r;
                if (row >= b->rows) break;
                const uint8_t *rp = b->W + (size_t)row * b->row_bytes;
                float sum[KC];
#pragma unroll
                for (uint32_t k = 0; k < KC; ++k) sum[k] = 0.0f;
                for (uint32_t c = 4u * lane; c < b->cols; c += 4u * KQ_WAVE) {
                    float wt[4];
                    weights_at<FMT>(rp, c, wt, malformed);
#pragma unroll
                    for (uint32_t k = 0; k < KC; ++k) {
                        if (k >= b->batch) break;
                        const float4 xv = *(const float4 *)(b->x + (size_t)k * b->cols + c);
                        sum[k] = fmaf(wt[0], xv.x, sum[k]);
                        sum[k] = fmaf(wt[1], xv.y, sum[k]);
                        sum[k] = fmaf(wt[2], xv.z, sum[k]);
                        sum[k] = fmaf(wt[3], xv.w, sum[k]);
                        if (k & 1u) __builtin_amdgcn_sched_barrier(0);
                    }
                }
#pragma unroll
                for (uint32_t k = 0; k < KC; ++k) {
                    float v = sum[k];
                    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, KQ_WAVE);
                    if (lane == 0u) part[(tile & 1u) * nw * (KC * 16u) + k * 16u + r] = v;
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            /* the other parity was read before the previous barrier */
            kq_lds_barrier();
            finish(tile, 1u);
        }
    } else {
        for (uint32_t tile = lo; tile < hi; ++tile) {
#pragma unroll
            for (uint32_t c = 0; c < NC; ++c, ++ent) {
                if (ent != 0u) {
                    const uint32_t after = n_ent - 1u - ent;
                    wait_after<IPW, kMaxPd - 1u>(after < a.pd - 1u ? after : a.pd - 1u);
                    kq_lds_barrier();
                }
                if (ent + a.pd < n_ent) issue();
                if (c == 0u && tile > lo) finish(tile - 1u, nw);
                const uint32_t u = c * nw + w;
                if (u < nu) { /* wave-uniform */
                    const uint32_t left = a.cols - kUnit * u;
                    const uint32_t live = PART && left < kUnit ? left / 32u : 8u;
                    const uint32_t at = w * UB + (FMT == KQ_LAUNCH_Q6_K ? (j * a.row_bytes) & 2u : 0u);
                    const uint32_t off = at & 2u;
                    const uint8_t *p = ring + slot * a.slot + j * a.pitch * 16u + at;
                    const f4 v = unit_product<FMT, M>(p, off, g, live, tile * kT + j < a.rows, A[c],
                                                      sums[c], malformed);
                    if constexpr (M == kQuad) {
                        /* the four parts of column g */
                        acc[0] += ldexpf(fmaf(0x1p-24f, v[2] + v[3], v[0] + v[1]), -sigs[u * KC + g]);
                    } else {
                        const int4 sg = *(const int4 *)(sigs + u * KC + 4u * (g & 1u));
                        const int at = M == kPair || g < 2u ? 0 : kTiny;
                        acc[0] += ldexpf(v[0], -sg.x - at);
                        acc[1] += ldexpf(v[1], -sg.y - at);
                        acc[2] += ldexpf(v[2], -sg.z - at);
                        acc[3] += ldexpf(v[3], -sg.w - at);
                    }
                }
                slot = slot == a.pd ? 0u : slot + 1u;
            }
            float *pw = part + ((tile & 1u) * nw + w) * (KC * 16u);
            if constexpr (M == kQuad) {
                pw[g * 16u + j] = acc[0];
                acc[0] = 0.0f;
            } else {
                /* columns 4g .. 4g + 3 of row j: operand rows 0 .. 7 and 8 .. 15 */
#pragma unroll
                for (uint32_t k = 0; k < 4u; ++k) {
                    const float o = acc[k] + __shfl_xor(acc[k], 32, KQ_WAVE);
                    if (g < 2u) pw[(4u * g + k) * 16u + j] = o;
                    acc[k] = 0.0f;
                }
            }
        }
        kq_lds_barrier();
        if (hi > lo) finish(hi - 1u, nw);
    }
    /* no LDS-DMA load may outlive the workgroup */
    wait_vm<0>();
    const MvtArgs *b = late_args();
    if (bad) kq_flag(b->status, KQ_DEV_INPUT);
    if (malformed) kq_flag(b->status, KQ_DEV_MALFORMED);
    if (nonfinite) kq_flag(b->status, KQ_DEV_NUMERIC);
    if (b->part_v != nullptr && t < KC * 16u) {
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) {
            const float ov = __shfl_xor(best_v, o, KQ_WAVE);
            const uint32_t oi = __shfl_xor(best_i, o, KQ_WAVE);
            argmax_merge(best_v, best_i, ov, oi);
        }
        if ((t & 15u) == 0u && (t >> 4) < b->batch) {
            const size_t row = (size_t)(t >> 4) * b->part_stride;
            b->part_v[row + blockIdx.x] = best_v;
            b->part_i[row + blockIdx.x] = best_i;
            for (uint32_t sl = blockIdx.x + gridDim.x; sl < b->part_stride; sl += gridDim.x) {
                b->part_v[row + sl] = -__builtin_inff();
                b->part_i[row + sl] = 0xffffffffu;
            }
        }
    }
}

/* ------------------------------------------------------------------ */
/* launch shape */

struct Plan {
    uint32_t nw, nc, pitch, slot, pd, lds, blocks;
};

uint32_t device_cus() {
    static uint32_t cus = 0u;
    if (cus == 0u) {
        int dev = 0, n = 0;
        cus = hipGetDevice(&dev) == hipSuccess &&
                      hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) ==
                          hipSuccess &&
                      n > 0
                  ? (uint32_t)n
                  : 256u;
    }
    return cus;
}

constexpr uint32_t kLdsCu = 160u * 1024u;
constexpr uint32_t kMaxEight = 2u; /* units per wave with two operands each */

/* The waves of a workgroup: the count (at most 10, 8 with more than two
 * operands of 32 registers each) that leaves the fewest idle in a row's last
 * chunk, the larger of equals: one unit a wave where a row has at most 10
 * (10240 x 2560 Q8_0 at 8 columns: 12.9 us with 10 waves of one unit, 22 with
 * 5 of two). Two workgroups per CU where their registers and two chunk slots
 * each fit (151936 x 2048 Q6_K at 4 columns: 61.8 us, 72.4 with one), and as
 * many slots as fit then. */
bool make_plan(uint32_t type, uint32_t rows, uint32_t cols, uint32_t batch, Plan &p) {
    const uint32_t ub = unit_bytes(type);
    if (ub == 0u || cols == 0u || cols % block_cols(type) != 0u) return false;
    const uint32_t nu = (cols + kUnit - 1u) / kUnit, ops = batch > 4u && is_binary32(type) ? 2u : 1u;
    const uint32_t kc = kCols;
    uint32_t best = 0u, best_idle = 0xffffffffu;
    for (uint32_t nw = 10u; nw >= 2u; --nw) {
        const uint32_t nc = (nu + nw - 1u) / nw;
        if (nc * ops > (ops == 2u ? 2u * kMaxEight : 5u) || (nc * ops > kNarrow && nw > 8u) || (nc > 3u && cols % kUnit != 0u)) continue;
        if (nc > 1u && (nw * ub) % 4u != 0u) continue; /* chunks start on dwords */
        const uint32_t idle = nc * nw - nu;
        if (idle < best_idle) {
            best = nw;
            best_idle = idle;
        }
    }
    if (best == 0u) return false;
    p.nw = best;
    p.nc = (nu + best - 1u) / best;
    const uint32_t units = (best * ub + 2u + 15u) / 16u;
    p.pitch = units | 1u;
    p.slot = (kT * p.pitch + 63u) / 64u * 1024u;
    const uint32_t fixed = 1024u + 2u * best * kc * 64u + p.nc * best * kc * 4u + best * 4u;
    /* per CU, by registers */
    const uint32_t waves = p.nc * ops == 1u ? 20u : p.nc * ops == 2u ? 12u : 8u;
    const uint32_t wgs = 2u * best <= waves && 2u * (2u * p.slot + fixed) <= kLdsCu ? 2u : 1u;
    uint32_t slots = (kLdsCu / wgs - fixed) / p.slot;
    if (slots > kMaxPd + 1u) slots = kMaxPd + 1u;
    if (slots < 2u) return false;
    p.pd = slots - 1u;
    p.lds = slots * p.slot + fixed;
    const uint32_t tiles = (rows + kT - 1u) / kT, resident = wgs * device_cus();
    p.blocks = tiles < resident ? tiles : resident;
    return true;
}

uint32_t row_bytes_of(uint32_t type, uint32_t cols) {
    return cols / block_cols(type) * (unit_bytes(type) / (kUnit / block_cols(type)));
}

template <uint32_t FMT, uint32_t NC, bool PART>
hipError_t launch_nc(const Plan &p, const MvtArgs &a, hipStream_t s) {
    constexpr Rows kMany = is_binary32(FMT) ? kEight : kPair;
    /* five units of four parts take longer to build (4000 x 10240 Q4_K, 2
     * columns: 18.7 us, kPair 16.4) */
    constexpr Rows kFew = NC >= 5u && kMany == kPair ? kPair : kQuad;
    const dim3 grid(p.blocks), block(p.nw * 64u);
    if (a.batch <= 4u) {
        hipLaunchKernelGGL((mv_tiles<FMT, NC, PART, kFew>), grid, block, p.lds, s, a);
    } else {
        if constexpr (kMany == kEight && NC > kMaxEight)
            return hipErrorInvalidValue;
        else
            hipLaunchKernelGGL((mv_tiles<FMT, NC, PART, kMany>), grid, block, p.lds, s, a);
    }
    return hipGetLastError();
}

template <uint32_t FMT>
hipError_t launch_fmt(const Plan &p, const MvtArgs &a, hipStream_t s) {
    if constexpr (block_cols(FMT) < kUnit) {
        if (a.cols % kUnit != 0u) {
            switch (p.nc) {
            case 1: return launch_nc<FMT, 1, true>(p, a, s);
            case 2: return launch_nc<FMT, 2, true>(p, a, s);
            case 3: return launch_nc<FMT, 3, true>(p, a, s);
            default: return hipErrorInvalidValue;
            }
        }
    }
    switch (p.nc) {
    case 1: return launch_nc<FMT, 1, false>(p, a, s);
    case 2: return launch_nc<FMT, 2, false>(p, a, s);
    case 3: return launch_nc<FMT, 3, false>(p, a, s);
    case 4: return launch_nc<FMT, 4, false>(p, a, s);
    case 5: return launch_nc<FMT, 5, false>(p, a, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

extern "C" int kq_launch_mv_tiles_supported(uint32_t type, uint32_t rows, uint32_t cols,
                                            uint32_t batch) {
    Plan p;
    if (batch < 1u || batch > kCols || !make_plan(type, rows, cols, batch, p)) return 0;
    /* rows of 34- and 18-byte blocks start on whole dwords (Q6_K ones may
     * not), and the last tile's offsets past the matrix stay within 32 bits */
    const uint64_t rb = row_bytes_of(type, cols);
    return (rb % 4u == 0u || type == KQ_LAUNCH_Q6_K) && rows * rb <= 0xffe00000ull;
}

extern "C" uint32_t kq_launch_mv_tiles_parts(uint32_t type, uint32_t rows, uint32_t cols,
                                             uint32_t batch) {
    Plan p;
    return make_plan(type, rows, cols, batch, p) ? p.blocks : 0u;
}

extern "C" hipError_t kq_launch_mv_tiles(uint32_t type, const void *W, uint32_t rows,
                                         uint32_t cols, const float *x, uint32_t batch, float *y,
                                         uint32_t *status, float *part_v, uint32_t *part_i,
                                         uint32_t part_stride, hipStream_t stream) {
    Plan p;
    if (!kq_launch_mv_tiles_supported(type, rows, cols, batch) || !make_plan(type, rows, cols, batch, p))
        return hipErrorInvalidValue;
    MvtArgs a;
    a.W = (const uint8_t *)W;
    a.rows = rows;
    a.cols = cols;
    a.row_bytes = row_bytes_of(type, cols);
    a.w_bytes = (rows * a.row_bytes + 3u) & ~3u;
    a.x = x;
    a.batch = batch;
    a.y = y;
    a.status = status;
    a.part_v = part_v;
    a.part_i = part_i;
    a.part_stride = part_stride;
    a.pitch = p.pitch;
    a.slot = p.slot;
    a.pd = p.pd;
    const uint32_t tiles = (rows + kT - 1u) / kT;
    a.tiles = tiles / p.blocks;
    a.more = tiles % p.blocks;
    switch (type) {
    case KQ_LAUNCH_Q4_K: return launch_fmt<KQ_LAUNCH_Q4_K>(p, a, stream);
    case KQ_LAUNCH_Q5_K: return launch_fmt<KQ_LAUNCH_Q5_K>(p, a, stream);
    case KQ_LAUNCH_Q6_K: return launch_fmt<KQ_LAUNCH_Q6_K>(p, a, stream);
    case KQ_LAUNCH_Q8_0: return launch_fmt<KQ_LAUNCH_Q8_0>(p, a, stream);
    case KQ_LAUNCH_Q5_1: return launch_fmt<KQ_LAUNCH_Q5_1>(p, a, stream);
    case KQ_LAUNCH_IQ4_NL: return launch_fmt<KQ_LAUNCH_IQ4_NL>(p, a, stream);
    default: return hipErrorInvalidValue;
    }
}
