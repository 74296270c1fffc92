/*
 * kq_mvtiles.hip — y = W x for 2 to 8 activation columns on the matrix
 * cores: GGUF Q4_K, Q5_K, Q6_K, Q8_0, Q5_1 and IQ4_NL rows.
 *
 * Restates the row loop of kq_weight_provider_linear_f32
 * (src/kq_weight_provider.c:464-475) for several activation vectors.
 *
 * The row engine (kq_rowdot.h) pays its dot per column: at four columns it
 * holds 4 x 32 activations a lane, and more than four take another launch
 * that reads the weights again. Here the weights are read and decoded once
 * for up to eight columns:
 *
 *   - One 16x16x32 fp16 step multiplies 16 weight rows by 16 operand rows:
 *     rows 0..7 hold the hi parts of the eight columns, rows 8..15 their lo
 *     parts (x = hi + lo to ~23 bits after an exact power-of-two scaling per
 *     column and 256-column unit), so one step serves all the columns.
 *   - A workgroup walks a contiguous run of 16-row tiles. A row is cut into
 *     units of 256 columns; wave w multiplies unit c nw + w of every row in
 *     the tile's c-th of NC chunks. Its activation operand, 32 registers a
 *     unit, is built once and stays in registers for the whole run.
 *   - A chunk (16 rows x nw units) is copied into an LDS ring by 16-byte
 *     LDS-DMA loads spread over the waves, PD chunks ahead of the one being
 *     multiplied. Rows sit at an odd pitch of 16-byte units, so the 16 rows
 *     a step reads hit distinct banks.
 *   - Each wave adds its hi and lo product rows and leaves 8 columns x 16
 *     rows in LDS; after the next barrier 128 threads add the waves in
 *     order, store, and keep the argmax partials: one per workgroup and
 *     column.
 *
 * Codes enter fp16 exactly. Q4_K and Q5_K fold the 6-bit sub-block scale
 * into the weight (at most 1953, exact) and take their mins off with one
 * small step against the columns' sub-block sums; Q6_K takes one 16x16x16
 * step per 16-column sub-block, the 32-weight formats one 16x16x32 step per
 * block, scaled in fp32.
 *
 * Bound: HBM for matrices that fill the device, the first loads' latency
 * and the operand's build below that. Against the row engine (and, for Q6_K
 * heads of 2 to 4 columns, the per-format matrix-core kernels that this one
 * replaced at equal times): 10240 x 2560 Q8_0 at 8 columns 76.7 -> 11.8 us
 * (2.4 TB/s), the 248320 x 2560 Q8_0 head at 5 columns 269 -> 140 us
 * (4.8 TB/s). Error against binary64 sums 0.8-1.5e-7 of the result in every
 * format (row engine 1.7-5.7e-7).
 */
#include "kq_launch.h"
#include "kq_device.h"
#include "kq_dma.h"
#include "kq_mfma.h"

namespace {

using namespace kq::mf;

constexpr uint32_t kT = 16;      /* rows per tile */
constexpr uint32_t kCols = 8;    /* activation columns */
constexpr uint32_t kMaxPd = 4;   /* chunks in flight, at most */

/* eight halves as four packed registers from here on: without the asm the
 * compiler keeps the unpacked values and packs them again at every use */
__device__ __forceinline__ h8 pinned(uint32_t x, uint32_t y, uint32_t z, uint32_t w) {
    asm volatile("" : "+v"(x), "+v"(y), "+v"(z), "+v"(w));
    return __builtin_bit_cast(h8, kq_u32x4{x, y, z, w});
}
/* the value of lane l ^ 8 (a rotation by 8 within the row of 16 lanes) */
__device__ __forceinline__ uint32_t ror8(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x128, 0xf, 0xf, true);
}
__device__ __forceinline__ float ror8(float x) { return __uint_as_float(ror8(__float_as_uint(x))); }
__device__ __forceinline__ uint32_t mag(float x) { return __float_as_uint(x) & 0x7fffffffu; }

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
 * 2^-5, sums 4g .. 4g + 3 on k-groups 0 and 1 (Q4_K, Q5_K); their block sums
 * times 2^-9 on k-groups 0 and 1 (against m) and times 16 2^-9 on 2 and 3
 * (against d, for the codes' middle 16) (Q5_1) */
constexpr bool has_min(uint32_t f) { return is_k(f) || f == KQ_LAUNCH_Q5_1; }

/* One unit of row j of the tile times the activation operand: returns
 * lane (j, g)'s products of operand rows 4g .. 4g + 3 in the operand's
 * scale. p: the unit's first byte in LDS (p - off is 4-byte aligned, off 0
 * or 2); live: steps that hold columns (8 but for
 * a row's last unit); real: row j exists. */
template <uint32_t FMT>
__device__ __forceinline__ f4 unit_product(const uint8_t *p, uint32_t off, uint32_t g,
                                           uint32_t live, bool real, const h8 (&A)[8], h4 sums,
                                           bool &malformed) {
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
    f4 acc = zero;
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
#pragma unroll
        for (uint32_t s = 0; s < 8u; ++s)
            acc = mfma32(A[s], sc.weights(s >> 2, g, dword_of(qa, qb, s & 3u, 0u), dword_of(qa, qb, s & 3u, 1u),
                                          dword_of(ha, hb, s & 3u, 0u), dword_of(ha, hb, s & 3u, 1u)),
                         acc);
        const uint32_t k01 = 0u - (uint32_t)(g < 2u);
        const f4 mm = mfma16(sums, byte_halves(k_mins(hd, g) & k01), zero);
        const f4 ss = mfma16(sums, byte_halves(k_scales(hd, g) & k01), zero);
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
                    const h8 &as = A[i >> 1];
                    const h4 a4 = (i & 1u) ? h4{as[4], as[5], as[6], as[7]}
                                           : h4{as[0], as[1], as[2], as[3]};
                    const h2 w0 = bytes_lo(c[k]) + bias, w1 = bytes_hi(c[k]) + bias;
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
        /* Q5_1 codes enter as q - 16; 16 d joins the min */
        const h2 bias = splat(FMT == KQ_LAUNCH_Q5_1 ? -1040.0f : -1152.0f);
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
                if (s < live)
                    mins[s & 3u] = (s >> 2) == (g & 1u) ? (g < 2u ? dm >> 16 : dm & 0xffffu)
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
                /* the 16 values (src/kq_numeric.c, IQ4_NL) plus 128 */
                auto look = [](uint32_t n) {
                    const uint32_t lo = __builtin_amdgcn_perm(0x766a5d4fu, 0x3f2d1801u, n & 0x07070707u);
                    const uint32_t hi = __builtin_amdgcn_perm(0xf1d9c5b5u, 0xa6998d81u, n & 0x07070707u);
                    const uint32_t b3 = (n >> 3) & 0x01010101u, m = (b3 << 8) - b3;
                    return (hi & m) | (lo & ~m);
                };
                c0 = look((q0 >> shn) & 0x0f0f0f0fu);
                c1 = look((q1 >> shn) & 0x0f0f0f0fu);
            }
            if (s >= live) d = 0.0f;
            const f4 t = mfma32(A[s], cat(bytes_lo(c0) + bias, bytes_hi(c0) + bias,
                                          bytes_lo(c1) + bias, bytes_hi(c1) + bias), zero);
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[k] = fmaf(d, t[k], acc[k]);
        }
        if constexpr (FMT == KQ_LAUNCH_Q5_1) {
            const h4 bm = __builtin_bit_cast(
                h4, make_uint2((mins[0] & 0xffffu) | (mins[1] << 16), (mins[2] & 0xffffu) | (mins[3] << 16)));
            const f4 mm = mfma16(sums, bm, zero);
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[k] = fmaf(0x1p9f, mm[k], acc[k]);
        }
        return acc;
    }
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
};

/* LDS-DMA instructions per wave and chunk: a chunk's 16 rows take at most
 * nw unit_bytes / 16 + 2 units each, 64 units an instruction, nw waves */
template <uint32_t FMT>
constexpr uint32_t ipw() {
    return (unit_bytes(FMT) + 32u + 63u) / 64u;
}

/* Register budget: 10 waves of up to 168 registers for one or two units a
 * wave, 8 of up to 256 for more. */
constexpr uint32_t kWideNc = 3u;
template <uint32_t NC>
constexpr int max_threads() {
    return NC < kWideNc ? 640 : 512;
}

/* PART: the row's last unit holds fewer than 256 columns */
template <uint32_t FMT, uint32_t NC, bool PART>
__global__ __launch_bounds__((max_threads<NC>())) void mv_tiles(MvtArgs a) {
    constexpr uint32_t UB = unit_bytes(FMT), IPW = ipw<FMT>();
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t nw = blockDim.x >> 6;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 15u, g = lane >> 4;
    /* ring, landing place of the padding loads, partial sums by tile parity
     * [2][nw][8][16], the units' powers of two [NC][nw][8] */
    uint8_t *ring = lds, *trash = ring + (a.pd + 1u) * a.slot;
    float *part = (float *)(trash + 1024u);
    int *sigs = (int *)(part + 2u * nw * 128u);

    const uint32_t ntiles = (a.rows + kT - 1u) / kT;
    const uint32_t lo = (uint32_t)((uint64_t)ntiles * blockIdx.x / gridDim.x);
    const uint32_t hi = (uint32_t)((uint64_t)ntiles * (blockIdx.x + 1u) / gridDim.x);
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
    if (n_ent != 0u) issue();

    /* the activation operand of this wave's units: lane (i, g) holds operand
     * row i, hi (i < 8) or lo of column i & 7. Lanes i and i + 8 split the
     * column's values between them (elements 0..3 and 4..7 of each step)
     * and trade their lo and hi halves: each value is scaled and split once
     * (768 -> 350 VALU instructions a unit, which the smallest products
     * feel). */
    h8 A[NC][8];
    h4 sums[NC];
    bool bad = false;
    {
        const uint32_t i = lane & 15u, col = i & 7u, half = i >> 3;
        /* columns past the row, and columns past the batch, read as zeros */
        const KqBuf bx = kq_buf(a.x, a.batch * a.cols * 4u);
        auto load = [&](uint32_t c, uint4 (&v)[8]) {
            const uint32_t u = c * nw + w, xo = (col * a.cols + kUnit * u) * 4u;
            const uint32_t left = u < nu && col < a.batch ? a.cols - kUnit * u : 0u;
#pragma unroll
            for (uint32_t s = 0; s < 8u; ++s) {
                const uint32_t at = half ? column_of<FMT>(g, s, 4u) : column_of<FMT>(g, s, 0u);
                v[s] = kq_ld128(bx, at < left ? xo + 4u * at : 0x80000000u, 0u);
            }
        };
        uint4 vn[8];
        load(0u, vn);
#pragma unroll
        for (uint32_t c = 0; c < NC; ++c) {
            float4 v[8];
#pragma unroll
            for (uint32_t s = 0; s < 8u; ++s) v[s] = __builtin_bit_cast(float4, vn[s]);
            if (c + 1u < NC) load(c + 1u, vn);
            uint32_t m = 0u; /* largest magnitude, as bits */
#pragma unroll
            for (uint32_t s = 0; s < 8u; ++s) {
                m = max(max(m, mag(v[s].x)), mag(v[s].y));
                m = max(max(m, mag(v[s].z)), mag(v[s].w));
            }
            m = max(m, ror8(m));
            m = max(m, (uint32_t)__shfl_xor(m, 16, KQ_WAVE));
            m = max(m, (uint32_t)__shfl_xor(m, 32, KQ_WAVE));
            /* largest magnitude into [2^14, 2^15); a column with a
             * non-finite value contributes zeros (the call fails) */
            const bool nf = m >= 0x7f800000u;
            bad |= nf;
            const int sig = !nf && m != 0u ? 15 - __builtin_amdgcn_frexp_expf(__uint_as_float(m)) : 0;
            if (g == 0u && i < kCols) sigs[(c * nw + w) * kCols + i] = sig;
            float run[2] = {0.0f, 0.0f}, blo[4], bhi[4];
#pragma unroll
            for (uint32_t s = 0; s < 8u; ++s) {
                if (nf) v[s] = float4{0.f, 0.f, 0.f, 0.f};
                const float xs[4] = {ldexpf(v[s].x, sig), ldexpf(v[s].y, sig), ldexpf(v[s].z, sig),
                                     ldexpf(v[s].w, sig)};
                h4 hv, lv;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    hv[e] = (_Float16)xs[e];
                    lv[e] = (_Float16)(xs[e] - (float)hv[e]);
                }
                const kq_u32x2 hb = __builtin_bit_cast(kq_u32x2, hv), lb = __builtin_bit_cast(kq_u32x2, lv);
                const uint32_t r0 = ror8(half ? hb.x : lb.x), r1 = ror8(half ? hb.y : lb.y);
                A[c][s] = pinned(half ? r0 : hb.x, half ? r1 : hb.y, half ? lb.x : r0, half ? lb.y : r1);
                if constexpr (has_min(FMT)) {
                    const float p = (xs[0] + xs[1]) + (xs[2] + xs[3]);
                    run[s >> 2] += p;
                    (s < 4u ? blo : bhi)[s & 3u] = p;
                }
            }
            float sm[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (is_k(FMT)) {
                /* lane (i, g) holds sub-blocks 2g and 2g + 1 */
                run[0] += ror8(run[0]);
                run[1] += ror8(run[1]);
                const int src = (int)(i + 32u * (g & 1u));
                sm[0] = __shfl(run[0], src, KQ_WAVE);
                sm[1] = __shfl(run[1], src, KQ_WAVE);
                sm[2] = __shfl(run[0], src + 16, KQ_WAVE);
                sm[3] = __shfl(run[1], src + 16, KQ_WAVE);
            } else if constexpr (FMT == KQ_LAUNCH_Q5_1) {
#pragma unroll
                for (uint32_t e = 0; e < 4u; ++e) {
                    blo[e] += ror8(blo[e]);
                    bhi[e] += ror8(bhi[e]);
                    blo[e] += __shfl_xor(blo[e], 16, KQ_WAVE);
                    bhi[e] += __shfl_xor(bhi[e], 16, KQ_WAVE);
                    blo[e] += __shfl_xor(blo[e], 32, KQ_WAVE);
                    bhi[e] += __shfl_xor(bhi[e], 32, KQ_WAVE);
                    sm[e] = (g & 1u) != 0u ? bhi[e] : blo[e];
                }
            }
            if constexpr (has_min(FMT)) {
#pragma unroll
                for (uint32_t e = 0; e < 4u; ++e) {
                    const float f = FMT == KQ_LAUNCH_Q5_1 ? sm[e] * (g < 2u ? 0x1p-9f : 0x1p-5f)
                                    : g < 2u              ? sm[e] * 0x1p-5f : 0.0f;
                    const _Float16 hv = (_Float16)f;
                    sums[c][e] = half ? (_Float16)(f - (float)hv) : hv;
                }
            } else {
                sums[c] = h4{};
            }
            /* one unit's values, and the next one's on their way */
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    for (uint32_t t = 1; t < a.pd && t < n_ent; ++t) issue();

    const uint32_t t = threadIdx.x; /* < 128: output column t / 16, row t % 16 */
    float best_v = -__builtin_inff();
    uint32_t best_i = 0xffffffffu;
    bool malformed = false, nonfinite = false;
    f4 acc = {0.f, 0.f, 0.f, 0.f};
    uint32_t slot = 0u, ent = 0u;
    auto finish = [&](uint32_t tile) {
        if (t < 128u) {
            const float *pp = part + (tile & 1u) * nw * 128u + t;
            float s = 0.0f;
            for (uint32_t q = 0; q < nw; ++q) s += pp[q * 128u];
            const uint32_t row = tile * kT + (t & 15u), col = t >> 4;
            if (row < a.rows && col < a.batch) {
                nonfinite |= !kq_isfinite(s);
                a.y[(size_t)col * a.rows + row] = s;
                argmax_merge(best_v, best_i, s, row);
            }
        }
    };
    for (uint32_t tile = lo; tile < hi; ++tile) {
#pragma unroll
        for (uint32_t c = 0; c < NC; ++c, ++ent) {
            /* this chunk's loads have landed (those of the chunks requested
             * after it may be in flight): in this wave, then in all */
            const uint32_t after = n_ent - 1u - ent;
            wait_after<IPW, kMaxPd - 1u>(after < a.pd - 1u ? after : a.pd - 1u);
            kq_lds_barrier();
            if (ent + a.pd < n_ent) issue();
            if (c == 0u && tile > lo) finish(tile - 1u);
            const uint32_t u = c * nw + w;
            if (u < nu) { /* wave-uniform */
                const uint32_t left = a.cols - kUnit * u;
                const uint32_t live = PART && left < kUnit ? left / 32u : 8u;
                const uint32_t at = w * UB + (FMT == KQ_LAUNCH_Q6_K ? (j * a.row_bytes) & 2u : 0u);
                const uint32_t off = at & 2u;
                const uint8_t *p = ring + slot * a.slot + j * a.pitch * 16u + at;
                const f4 v = unit_product<FMT>(p, off, g, live, tile * kT + j < a.rows, A[c],
                                               sums[c], malformed);
                const int4 sg = *(const int4 *)(sigs + u * kCols + 4u * (g & 1u));
                acc[0] += ldexpf(v[0], -sg.x);
                acc[1] += ldexpf(v[1], -sg.y);
                acc[2] += ldexpf(v[2], -sg.z);
                acc[3] += ldexpf(v[3], -sg.w);
            }
            slot = slot == a.pd ? 0u : slot + 1u;
        }
        /* columns 4g .. 4g + 3 of row j: the hi and the lo product rows */
        float *pw = part + ((tile & 1u) * nw + w) * 128u;
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            const float o = acc[k] + __shfl_xor(acc[k], 32, KQ_WAVE);
            if (g < 2u) pw[(4u * g + k) * 16u + j] = o;
            acc[k] = 0.0f;
        }
    }
    kq_lds_barrier();
    if (hi > lo) finish(hi - 1u);
    /* no LDS-DMA load may outlive the workgroup */
    wait_vm<0>();
    if (bad) kq_flag(a.status, KQ_DEV_INPUT);
    if (malformed) kq_flag(a.status, KQ_DEV_MALFORMED);
    if (nonfinite) kq_flag(a.status, KQ_DEV_NUMERIC);
    if (a.part_v != nullptr && t < 128u) {
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) {
            const float ov = __shfl_xor(best_v, o, KQ_WAVE);
            const uint32_t oi = __shfl_xor(best_i, o, KQ_WAVE);
            argmax_merge(best_v, best_i, ov, oi);
        }
        if ((t & 15u) == 0u && (t >> 4) < a.batch) {
            const size_t row = (size_t)(t >> 4) * a.part_stride;
            a.part_v[row + blockIdx.x] = best_v;
            a.part_i[row + blockIdx.x] = best_i;
            for (uint32_t sl = blockIdx.x + gridDim.x; sl < a.part_stride; sl += gridDim.x) {
                a.part_v[row + sl] = -__builtin_inff();
                a.part_i[row + sl] = 0xffffffffu;
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

/* The waves of a workgroup: the count (at most 10, 8 with three or more
 * units each) that leaves the fewest idle in a row's last chunk, the larger
 * of equals: one unit a wave where a row has at most 10 (10240 x 2560 Q8_0
 * at 8 columns: 12.9 us with 10 waves of one unit, 22 with 5 of two). Two
 * workgroups per CU where their registers and two chunk slots each fit
 * (151936 x 2048 Q6_K at 4 columns: 61.8 us, 72.4 with one), and as many
 * slots as fit then. */
bool make_plan(uint32_t type, uint32_t rows, uint32_t cols, Plan &p) {
    const uint32_t ub = unit_bytes(type);
    if (ub == 0u || cols == 0u || cols % block_cols(type) != 0u) return false;
    const uint32_t nu = (cols + kUnit - 1u) / kUnit;
    uint32_t best = 0u, best_idle = 0xffffffffu;
    for (uint32_t nw = 10u; nw >= 2u; --nw) {
        const uint32_t nc = (nu + nw - 1u) / nw;
        if (nc > 5u || (nc >= kWideNc && nw > 8u) || (nc > 3u && cols % kUnit != 0u)) continue;
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
    const uint32_t fixed = 1024u + 2u * best * 512u + p.nc * best * kCols * 4u;
    const uint32_t waves = p.nc == 1u ? 20u : p.nc < kWideNc ? 12u : 8u; /* per CU, by registers */
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
    hipLaunchKernelGGL((mv_tiles<FMT, NC, PART>), dim3(p.blocks), dim3(p.nw * 64u), p.lds, s, a);
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
    if (batch < 1u || batch > kCols || !make_plan(type, rows, cols, p)) return 0;
    /* rows of 34- and 18-byte blocks start on whole dwords (Q6_K ones may
     * not), and the last tile's offsets past the matrix stay within 32 bits */
    const uint64_t rb = row_bytes_of(type, cols);
    return (rb % 4u == 0u || type == KQ_LAUNCH_Q6_K) && rows * rb <= 0xffe00000ull;
}

extern "C" uint32_t kq_launch_mv_tiles_parts(uint32_t type, uint32_t rows, uint32_t cols) {
    Plan p;
    return make_plan(type, rows, cols, p) ? p.blocks : 0u;
}

extern "C" hipError_t kq_launch_mv_tiles(uint32_t type, const void *W, uint32_t rows,
                                         uint32_t cols, const float *x, uint32_t batch, float *y,
                                         uint32_t *status, float *part_v, uint32_t *part_i,
                                         uint32_t part_stride, hipStream_t stream) {
    Plan p;
    if (!kq_launch_mv_tiles_supported(type, rows, cols, batch) || !make_plan(type, rows, cols, p))
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
