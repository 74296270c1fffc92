/*
 * kq_gemm.hip — the prefill expert products for many tokens per expert:
 * gate/up + SwiGLU and down, up to 64 tokens against one decode of the
 * weights.
 *
 * The reference forms every (token, selected expert) pair's products one
 * token at a time (src/kq_moe_qwen38.c:722-765 via
 * kq_weight_provider_linear_f32, src/kq_weight_provider.c:378-509). The
 * 16-token passes (kq_grouped_gu.hip, kq_grouped_dn.hip) read and decode an
 * expert's rows once per 16 of its tokens; with 49 tokens per expert that is
 * four times, and decoding bounds them. Here one work item is up to 64
 * tokens of an expert:
 *
 *   - A workgroup of eight waves multiplies 64 tokens by 256 weight rows,
 *     32 rows (two 16-row tiles) per wave, so every weight is decoded once
 *     per item, in registers. Per 16 x 16 tile and 32 columns: one
 *     16x16x32 MFMA each for the activations' hi and lo halves.
 *   - The tokens' split rows come through a double-buffered LDS image,
 *     gathered by LDS-DMA, one barrier per step (256 columns for the K
 *     formats, 128 for the others). A row's 16-byte units are permuted by
 *     its low bits, so the 16 rows of a fragment hit distinct banks.
 *   - K-format rows go straight to registers one step ahead: a lane reads
 *     the 32 bytes it multiplies. The other formats' bytes are small pieces
 *     shared by lanes, and come through a per-wave LDS slot.
 *   - Fragments of 16 tokens that an item does not have are not loaded or
 *     multiplied.
 *   - The workgroups of a die walk an equal, contiguous range of the (item,
 *     row tile) sequence side by side, so an item's tokens come to its L2
 *     once; the loads run one step ahead across tiles.
 *
 * Measured at 2499 tokens, 512 experts, 10 per token, 2560 x 640, against the
 * 16-token passes: gate/up Q4_K 779 -> 587 us, down Q5_1 592 -> 510 us, the Q8_0
 * shared expert (as 64-token items of a dense product) 332 -> 133 us. Error of
 * the layer against binary64 1.09e-6, as theirs. What bounds it: the matrix cores
 * are busy for 31 % and 18 % of that, the vector ALU (decode, scales) about as
 * long, and with two waves of 250 registers per SIMD the two overlap little;
 * sixteen waves of one tile each (128 registers, spilled) took 771 us for the
 * down product.
 */
#include "kq_launch.h"
#include "kq_device.h"
#include "kq_dma.h"
#include "kq_mfma.h"
#include "kq_stage.h"

#include <type_traits>

namespace {

using namespace kq::mf;

constexpr uint32_t kM = 64;       /* tokens per item */
constexpr uint32_t kDies = 8;     /* workgroups go round-robin over the dies */
constexpr uint32_t kShared = 0x80000000u;
constexpr uint32_t kOut = 0x80000000u; /* an offset past every buffer */
/* Steps (of 128 columns) whose products a sum takes; the output holds the sum
 * of the runs before. The shared expert's 2560 columns in one sum err by 3.0e-7
 * of its output, in four by 2.2e-7, as in dense_q8's parts (two: 2.4e-7); 24
 * us more of the 2499-token layer. The K formats' few blocks are one sum. */
constexpr uint32_t kRun = 5;

/* a wave-uniform dword written by an earlier launch */
__device__ __forceinline__ uint32_t uniform(const uint32_t *p) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)*p);
}

/* a value loaded a step ago, from the lane whose address is turn. The asm
 * keeps every use behind this point: moved up to where the load was issued,
 * one would wait for it there. */
__device__ __forceinline__ uint4 arrived(uint4 v, uint32_t turn) {
    asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w));
    auto get = [&](uint32_t x) {
        return (uint32_t)__builtin_amdgcn_ds_bpermute((int)turn, (int)x);
    };
    return make_uint4(get(v.x), get(v.y), get(v.z), get(v.w));
}

struct GmArgs {
    const uint8_t *w0, *w1;   /* gate and up, or the one matrix (routed stacks) */
    const uint8_t *s0, *s1;   /* the same of the shared expert */
    const _Float16 *xh, *xl;  /* split activations [src_rows][k] */
    const _Float16 *sx;       /* their sub-block sums (kq_stage.h), K formats */
    const int *sig;
    const uint32_t *perm_tok; /* source row of a routed position; null: itself */
    const uint32_t *items;    /* [n][2]: expert | kShared, first | count << 24 */
    const uint32_t *n_items;
    uint32_t src_rows, pairs; /* pairs: tokens * top_k, the first shared position */
    uint32_t rows, k;
    float *out;               /* [positions][stride] */
    uint32_t stride;
    uint32_t plain;           /* items null: tokens of w0 and s0, side by side in out */
    uint32_t *status;
};

/* LDS image and weight slot of one step */
template <uint32_t FMT, uint32_t NW, uint32_t NT>
struct GmShape {
    static constexpr bool K = is_k(FMT);
    static constexpr uint32_t COLS = K ? 256u : 128u;
    static constexpr uint32_t UR = COLS / 8u;             /* 16-byte units per row */
    static constexpr uint32_t HALF = kM * COLS * 2u;       /* the hi rows; lo follow */
    static constexpr uint32_t RPI = 64u / UR;              /* rows per instruction */
    static constexpr uint32_t RPQ = NW / 2u * RPI;         /* rows by one load of every wave */
    static constexpr uint32_t NQ = kM / RPQ;               /* a wave's loads */
    static constexpr uint32_t IMG = 2u * HALF + (K ? 2048u : 0u);
    /* per row of a step: units of weight bytes */
    static constexpr uint32_t UPR = K ? 0u : FMT == KQ_LAUNCH_Q5_1 ? 6u : FMT == KQ_LAUNCH_Q8_0 ? 9u : 10u;
    static constexpr uint32_t WI = (16u * NT * UPR + 63u) / 64u;
    static constexpr uint32_t SLOT = WI * 1024u;           /* per wave */
    static constexpr uint32_t MINS = FMT == KQ_LAUNCH_Q5_1 ? 8u * kM * 16u : 0u; /* 8 steps */
    static constexpr uint32_t LDS = 2u * IMG + 2u * NW * SLOT + 2u * MINS + 2u * kM * 4u;
    static_assert(LDS <= 160u * 1024u, "LDS");
    /* The 16-byte unit of a row's step that lane k-group g multiplies in MFMA
     * step s. K formats: a lane reads bytes 16 g .. + 15 of each half of qs,
     * so steps 0..3 are columns 16 (g & 1) .. of sub-blocks 2 (g >> 1), + 1
     * and steps 4..7 the same of sub-blocks 4 + 2 (g >> 1), + 1. */
    __device__ __forceinline__ static constexpr uint32_t unit(uint32_t g, uint32_t s) {
        return K ? 16u * (s >> 2) + 8u * (g >> 1) + 4u * ((s >> 1) & 1u) + 2u * (g & 1u) + (s & 1u)
                 : 4u * s + g;
    }
    /* Where unit u of row r is kept, and back. A 16-byte read takes 16 lanes a
     * cycle, of neighbouring k-groups for different rows: their units share
     * one 16-unit column, permuted by the row. */
    __device__ __forceinline__ static uint32_t place(uint32_t u, uint32_t r) {
        if constexpr (!K) return u ^ (r & 15u);
        return 8u * (u & 2u) + (((u & 1u) + ((u >> 1) & 14u)) ^ (r & 15u));
    }
    __device__ __forceinline__ static uint32_t source_unit(uint32_t p, uint32_t r) {
        const uint32_t v = (p & 15u) ^ (r & 15u);
        if constexpr (!K) return v;
        return ((p >> 3) & 2u) + (v & 1u) + 2u * (v & 14u);
    }
    /* the byte that step s flips in the place of step 0's unit */
    __device__ __forceinline__ static constexpr uint32_t flip(uint32_t s) {
        return 16u * (K ? (s & 3u) + 2u * (s & 4u) : 4u * s);
    }
};

/* The matrices' rows a wave multiplies: GU, 16 gate rows and the same 16 up
 * rows of a tile of 128; otherwise 32 rows of a tile of 256. */
template <uint32_t FMT, bool GU, uint32_t NW, uint32_t NT>
__global__ __launch_bounds__(NW * 64) void gm_product(GmArgs a) {
    using S = GmShape<FMT, NW, NT>;
    static_assert(GU == S::K && (!GU || NT == 2u), "gate/up pairs in the K formats");
    constexpr bool Q5 = FMT == KQ_LAUNCH_Q5_K;
    constexpr uint32_t UB = unit_bytes(FMT), QS = Q5 ? 48u : 16u;
    constexpr uint32_t TROWS = GU ? 16u * NW : 16u * NT * NW;
    __shared__ __align__(16) uint8_t lds[S::LDS];
    uint8_t *slots = lds + 2u * S::IMG;
    uint8_t *msum = slots + 2u * NW * S::SLOT;
    int *s_sig = (int *)(msum + 2u * S::MINS);

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 15u, g = lane >> 4;
    const uint32_t steps = a.k / S::COLS;
    const uint32_t rb = a.k / 256u * UB + (a.k & 128u) / 128u * (UB / 2u); /* row bytes */
    const uint32_t wbytes = a.rows * rb;
    const uint32_t nt = (a.rows + TROWS - 1u) / TROWS;
    const uint32_t chunks = (a.src_rows + kM - 1u) / kM;
    const uint32_t n_items = a.plain ? a.plain * chunks : uniform(a.n_items);
    const uint64_t total = (uint64_t)n_items * nt;
    /* die x of kDies walks an equal, contiguous range of the tiles, its
     * workgroups side by side */
    const uint32_t die = blockIdx.x % kDies, peers = gridDim.x / kDies;
    const uint32_t lo = (uint32_t)(total * die / kDies) + blockIdx.x / kDies;
    const uint32_t hi = (uint32_t)(total * (die + 1u) / kDies);
    if (lo >= hi) return;

    struct Item {
        uint32_t ex, first, count;
    };
    auto item = [&](uint32_t it) {
        if (a.plain) {
            const uint32_t c = it / a.plain;
            return Item{(it - c * a.plain) ? kShared : 0u, c * kM, (uint32_t)min(a.src_rows - c * kM, kM)};
        }
        const uint32_t ex = uniform(a.items + 2u * it), fc = uniform(a.items + 2u * it + 1u);
        return Item{ex, fc & 0xffffffu, fc >> 24};
    };

    /* ---- requests: item, tile and step asked for next ---- */
    const uint32_t xbytes = a.src_rows * a.k * 2u;
    const kq_i4v bh = dma_rsrc(a.xh, xbytes), bl = dma_rsrc(a.xl, xbytes);
    const bool low = (w & 1u) != 0u; /* odd waves fetch the lo rows */
    const kq_i4v bx = {__builtin_amdgcn_readfirstlane(low ? bl.x : bh.x),
                       __builtin_amdgcn_readfirstlane(low ? bl.y : bh.y),
                       __builtin_amdgcn_readfirstlane(low ? bl.z : bh.z),
                       __builtin_amdgcn_readfirstlane(low ? bl.w : bh.w)};
    const kq_i4v bs = dma_rsrc(a.sx, S::K ? a.src_rows * (a.k / 128u) * 16u : 0u);
    const KqBuf bperm = kq_buf(a.perm_tok, a.perm_tok != nullptr ? a.pairs * 4u : 0u);
    const KqBuf bsig = kq_buf(a.sig, a.src_rows * 4u);
    uint32_t r_t = lo, r_it = lo / nt, r_tile = lo - r_it * nt, r_step = 0u, r_nf = 0u, r_par = 1u;
    bool r_new = true;
    uint32_t xo[S::NQ], so = kOut;
    const uint8_t *m0 = nullptr, *m1 = nullptr;
    /* the next step's K-format rows: four neighbouring lanes of one row, for
     * whole 64-byte requests (row j in lanes j, j + 16, .. took 64 requests a
     * load); turned into MFMA's order on arrival */
    uint4 nhd[2], nqa[2], nqb[2], nqh[2];
    const uint32_t turn = 4u * (4u * j + g);

    /* this lane's unit of the wave's rows in each of its loads: row (past
     * them: none), byte. Q6_K: half n of a block (from the dword it starts in)
     * is 5 units of ql, 3 of qh, 2 of scales and d; wn what half 1 adds. */
    constexpr uint32_t WI = S::K ? 1u : S::WI, UPR = S::K ? 1u : S::UPR;
    uint32_t wr[WI], wo[WI], wn[WI];
#pragma unroll
    for (uint32_t q = 0; q < WI; ++q) {
        const uint32_t u = 64u * q + lane, c = u % UPR;
        wr[q] = u / UPR < 16u * NT ? u / UPR : kOut;
        wo[q] = u / UPR * rb;
        if constexpr (FMT == KQ_LAUNCH_Q6_K) {
            wo[q] += c < 5u ? 16u * c : c < 8u ? 128u + 16u * (c - 5u) : 192u + 16u * (c - 8u);
            wn[q] = c < 5u ? 64u : c < 8u ? 32u : 8u;
        } else {
            wo[q] += 16u * c;
        }
    }
    auto new_item = [&]() {
        const Item it = item(r_it);
        const bool sh = (it.ex & kShared) != 0u;
        m0 = sh ? a.s0 : a.w0 + (size_t)it.ex * wbytes;
        m1 = sh ? a.s1 : a.w1 + (size_t)it.ex * wbytes;
        r_nf = (it.count + 15u) / 16u;
        r_par ^= 1u;
        const bool perm = a.perm_tok != nullptr && !sh;
        const uint32_t base = sh && a.perm_tok == nullptr && !a.plain ? a.pairs + it.first : it.first;
        /* every list entry this lane needs, then the rows they name */
        constexpr uint32_t NQ = S::NQ;
        auto entry = [&](uint32_t r) {
            return kq_ld32(bperm, perm && r < it.count ? (it.first + r) * 4u : kOut, 0u);
        };
        auto source = [&](uint32_t r, uint32_t listed) {
            const uint32_t t = perm ? listed : base + r;
            return r < it.count && t < a.src_rows ? t : kOut;
        };
        uint32_t le[NQ], ls = 0u;
#pragma unroll
        for (uint32_t q = 0; q < NQ; ++q) le[q] = entry(S::RPQ * q + S::RPI * (w >> 1) + lane / S::UR);
        if constexpr (S::K) ls = entry((32u * w + (lane >> 1)) & 63u);
        const uint32_t ll = entry(lane);
#pragma unroll
        for (uint32_t q = 0; q < NQ; ++q) {
            const uint32_t r = S::RPQ * q + S::RPI * (w >> 1) + lane / S::UR;
            const uint32_t t = source(r, le[q]);
            xo[q] = t != kOut ? t * a.k * 2u + 16u * S::source_unit(lane & (S::UR - 1u), r) : kOut;
        }
        if constexpr (S::K) {
            const uint32_t t = source((32u * w + (lane >> 1)) & 63u, ls);
            so = t != kOut ? t * (a.k / 128u) * 16u + 16u * (lane & 1u) : kOut;
        }
        if (w == 0u) {
            const uint32_t t = source(lane, ll);
            s_sig[r_par * kM + lane] = (int)kq_ld32(bsig, t != kOut ? t * 4u : kOut, 0u);
        }
        if constexpr (S::MINS != 0u) {
            /* the 32-column sums of every token, times 2^-5, hi + lo: the
             * operand of the min term */
            const KqBuf ch = kq_buf(a.xh, xbytes), cl = kq_buf(a.xl, xbytes);
            const uint32_t t = source(lane, ll);
            for (uint32_t b = w; b < a.k / 32u; b += NW) {
                float v = 0.0f;
#pragma unroll
                for (uint32_t u = 0; u < 4u; ++u) {
                    const uint32_t o = t != kOut ? (t * a.k + 32u * b + 8u * u) * 2u : kOut;
                    const h8 hh = __builtin_bit_cast(h8, kq_ld128(ch, o, 0u));
                    const h8 ll = __builtin_bit_cast(h8, kq_ld128(cl, o, 0u));
#pragma unroll
                    for (int e = 0; e < 8; ++e) v += (float)hh[e] + (float)ll[e];
                }
                v *= 0.03125f;
                const _Float16 vh = (_Float16)v;
                _Float16 *d = (_Float16 *)(msum + r_par * S::MINS + ((b >> 2) * kM + lane) * 16u);
                d[b & 3u] = vh;
                d[4u + (b & 3u)] = (_Float16)(v - (float)vh);
            }
        }
    };
    auto request = [&](uint32_t buf) {
        if (r_new) {
            r_new = false;
            new_item();
        }
        const uint32_t img = lds_addr(lds) + buf * S::IMG;
        if constexpr (S::K) {
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const KqBuf bw = kq_buf(m == 1 ? m1 : m0, wbytes);
                const uint32_t row = r_tile * TROWS + 16u * w + (lane >> 2);
                const uint32_t o = row < a.rows ? row * rb : kOut, st = r_step * UB;
                nhd[m] = kq_ld128(bw, o, st);
                nqa[m] = kq_ld128(bw, o + QS + 16u * (lane & 3u), st);
                nqb[m] = kq_ld128(bw, o + QS + 64u + 16u * (lane & 3u), st);
                if constexpr (Q5) nqh[m] = kq_ld128(bw, o + 16u + 16u * (lane & 1u), st);
            }
            if (w < 2u) dma16(bs, so + 32u * r_step, img + 2u * S::HALF + 1024u * w);
        } else {
            const kq_i4v bw = dma_rsrc(m0, wbytes);
            const kq_i4v rw = {__builtin_amdgcn_readfirstlane(bw.x), __builtin_amdgcn_readfirstlane(bw.y),
                               __builtin_amdgcn_readfirstlane(bw.z), __builtin_amdgcn_readfirstlane(bw.w)};
            const uint32_t dst = lds_addr(slots) + (buf * NW + w) * S::SLOT;
            const uint32_t row0 = r_tile * TROWS + 16u * NT * w;
            const uint32_t tile = row0 * rb, left = a.rows > row0 ? a.rows - row0 : 0u;
#pragma unroll
            for (uint32_t q = 0; q < S::WI; ++q) {
                uint32_t in = wo[q];
                if constexpr (FMT == KQ_LAUNCH_Q6_K)
                    in += ((r_step >> 1) * UB & ~3u) + (r_step & 1u ? wn[q] : 0u);
                else
                    in += r_step * (UB / 2u);
                dma16(rw, wr[q] < left ? tile + in : kOut, dst + 1024u * q);
            }
        }
        const uint32_t dst = __builtin_amdgcn_readfirstlane(img + (low ? S::HALF : 0u) + (w >> 1) * 1024u);
#pragma unroll
        for (uint32_t q = 0; q < S::NQ; ++q)
            if (q * S::RPQ < 16u * r_nf)
                dma16(bx, xo[q] + r_step * S::COLS * 2u, dst + 1024u * (NW / 2u) * q);
        if (++r_step == steps) {
            r_step = 0u;
            r_t += peers;
            r_tile += peers;
            if (r_tile >= nt) {
                r_it = r_t / nt;
                r_tile = r_t - r_it * nt;
                r_new = true;
            }
        }
    };

    /* ---- products ---- */
    /* (Q5_1: in 2^-5 of the others' scale, that of the sums the min term adds) */
    f4 acc[NT][4];
    auto clear = [&]() {
#pragma unroll
        for (uint32_t m = 0; m < NT; ++m)
#pragma unroll
            for (int f = 0; f < 4; ++f) acc[m][f] = f4{0.f, 0.f, 0.f, 0.f};
    };
    clear();
    bool bad = false, malformed = false;
    /* the 32-column formats' many scales: 0, or NaN once a scale was not finite: one multiply-add a pair of them */
    h2 finite = splat(0.0f);
    auto check = [&](uint32_t pair) { finite = fma2(as_h2(pair), splat(0.0f), finite); };
    uint32_t c_t = lo, c_tile = lo % nt, c_step = 0u, c_run = 0u, par = 0u;
    Item cur = item(lo / nt);
    uint4 hd[2], qa[2], qb[2], qh[2] = {};

    /* one step of NF fragments; img: the step's activations, slot: this
     * wave's weight bytes */
    auto product = [&](auto nf_tag, const uint8_t *img, const uint8_t *slot) {
        constexpr uint32_t NF = decltype(nf_tag)::value;
        const f4 zero = {0.f, 0.f, 0.f, 0.f};
        if constexpr (S::K) {
            /* pairs of sub-blocks g >> 1 (steps 0..3) and 2 + (g >> 1) */
            const uint32_t pr[2] = {g >> 1, 2u + (g >> 1)};
            const KPair<FMT, false> sc[2][2] = {{{hd[0], pr[0]}, {hd[0], pr[1]}},
                                                {{hd[1], pr[0]}, {hd[1], pr[1]}}};
            auto weights = [&](uint32_t m, uint32_t s) {
                const uint4 &q = (s >> 2) ? qb[m] : qa[m];
                return sc[m][s >> 2].weights((s >> 1) & 1u, pr[s >> 2], (s & 1u) ? q.z : q.x,
                                             (s & 1u) ? q.w : q.y, (s & 1u) ? qh[m].z : qh[m].x,
                                             (s & 1u) ? qh[m].w : qh[m].y);
            };
            f4 t[2][NF];
#pragma unroll
            for (uint32_t f = 0; f < NF; ++f) t[0][f] = t[1][f] = zero;
            const uint32_t p0 = j * (S::COLS * 2u) + 16u * S::place(S::unit(g, 0u), j);
            /* per step the hi halves of every fragment, then the lo halves (a
             * tile's next product waits for its last), read two ahead */
            h8 ah[2], al[2], b0, b1;
            auto read = [&](uint32_t i) {
                const uint8_t *p = img + (p0 ^ S::flip(i / NF)) + i % NF * 16u * S::COLS * 2u;
                ah[i & 1u] = *(const h8 *)p;
                al[i & 1u] = *(const h8 *)(p + S::HALF);
            };
            read(0u);
#pragma unroll
            for (uint32_t i = 0; i < 8u * NF; ++i) {
                const uint32_t s = i / NF, f = i % NF;
                if (f == 0u) {
                    b0 = weights(0u, s);
                    b1 = weights(1u, s);
                }
                if (i + 1u < 8u * NF) read(i + 1u);
                t[0][f] = mfma32(ah[i & 1u], b0, t[0][f]);
                t[1][f] = mfma32(ah[i & 1u], b1, t[1][f]);
                t[0][f] = mfma32(al[i & 1u], b0, t[0][f]);
                t[1][f] = mfma32(al[i & 1u], b1, t[1][f]);
                /* the next fragment's reads before this one's products */
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
            }
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const float d = half_bits(hd[m].x), dmin = half_bits(hd[m].x >> 16);
                malformed |= !kq_isfinite(d) || !kq_isfinite(dmin);
                const float dw = d * 0x1p14f, dm = dmin * -32.0f; /* the sums carry 2^-5 */
                /* k-groups 0, 1 the sums' hi halves, 2, 3 the lo halves */
                const h4 mins = byte_halves(k_mins(hd[m], g & 1u));
                const uint8_t *p = img + 2u * S::HALF + j * 32u + 16u * (g & 1u) + 8u * (g >> 1);
#pragma unroll
                for (uint32_t f = 0; f < NF; ++f) {
                    const f4 mm = mfma16(*(const h4 *)(p + 512u * f), mins, zero);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[m][f][e] += fmaf(dw, t[m][f][e], dm * mm[e]);
                }
            }
        } else if constexpr (FMT == KQ_LAUNCH_Q6_K) {
            const h2 bias = splat(-1056.0f); /* 1024 + 32 */
            const uint32_t off = ((c_step >> 1) & 1u) * 2u, n = c_step & 1u;
            const uint32_t *wr[NT];
            float d[NT];
            uint32_t sc[NT][2];
#pragma unroll
            for (uint32_t m = 0; m < NT; ++m) {
                wr[m] = (const uint32_t *)(slot + (16u * m + j) * (S::UPR * 16u));
                const uint32_t dd = wr[m][32u + (n ? 2u : 4u)];
                d[m] = half_bits(off ? dd >> 16 : dd);
                check((off ? dd >> 16 : dd) & 0xffffu);
                sc[m][0] = kq_align2(wr[m][33], wr[m][32], off);
                sc[m][1] = kq_align2(wr[m][34], wr[m][33], off);
            }
#pragma unroll
            for (uint32_t h = 0; h < 2u; ++h) {
                uint32_t c[NT][4];
#pragma unroll
                for (uint32_t m = 0; m < NT; ++m) {
                    const uint32_t *wg = wr[m] + g;
                    const uint32_t x = kq_align2(wg[4u * h + 1u], wg[4u * h], off);
                    const uint32_t y = kq_align2(wg[4u * h + 9u], wg[4u * h + 8u], off);
                    const uint32_t z = kq_align2(wg[4u * h + 21u], wg[4u * h + 20u], off);
                    c[m][0] = (x & 0x0f0f0f0fu) | ((z << 4) & 0x30303030u);
                    c[m][1] = (y & 0x0f0f0f0fu) | ((z << 2) & 0x30303030u);
                    c[m][2] = ((x >> 4) & 0x0f0f0f0fu) | (z & 0x30303030u);
                    c[m][3] = ((y >> 4) & 0x0f0f0f0fu) | ((z >> 2) & 0x30303030u);
                }
#pragma unroll
                for (uint32_t k = 0; k < 4u; ++k) {
                    const uint32_t sub = 2u * k + h;
                    h4 b[NT];
                    float ds[NT];
#pragma unroll
                    for (uint32_t m = 0; m < NT; ++m) {
                        const h2 x = bytes_lo(c[m][k]) + bias, y = bytes_hi(c[m][k]) + bias;
                        b[m] = h4{x.x, x.y, y.x, y.y};
                        ds[m] = d[m] * (float)(int8_t)((sc[m][sub >> 2] >> (8u * (sub & 3u))) & 0xffu);
                    }
                    const uint8_t *p = img + j * (S::COLS * 2u) +
                                       16u * S::place(4u * k + 2u * h + (g >> 1), j) + 8u * (g & 1u);
#pragma unroll
                    for (uint32_t f = 0; f < NF; ++f) {
                        const h4 ah = *(const h4 *)(p + f * 16u * S::COLS * 2u);
                        const h4 al = *(const h4 *)(p + f * 16u * S::COLS * 2u + S::HALF);
#pragma unroll
                        for (uint32_t m = 0; m < NT; ++m) {
                            const f4 t = mfma16(al, b[m], mfma16(ah, b[m], zero));
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                acc[m][f][e] = fmaf(ds[m], t[e], acc[m][f][e]);
                        }
                    }
                }
            }
        } else {
            /* Q5_1 codes are unsigned, Q8_0 ones offset by 128 */
            constexpr bool Q51 = FMT == KQ_LAUNCH_Q5_1;
            const h2 bias = splat(Q51 ? -1024.0f : -1152.0f);
            const uint32_t shn = g >= 2u ? 4u : 0u;
            uint32_t mins[NT][4];
            const uint32_t p0 = j * (S::COLS * 2u) + 16u * S::place(S::unit(g, 0u), j);
            h8 x[3], b[NT];
            float d[NT];
            auto read = [&](uint32_t i) {
                x[i % 3u] = *(const h8 *)(img + (p0 ^ S::flip(i / (2u * NF))) +
                                          (i / NF % 2u) * S::HALF + i % NF * 16u * S::COLS * 2u);
            };
            auto decode = [&](uint32_t s) {
#pragma unroll
                for (uint32_t m = 0; m < NT; ++m) {
                    const uint32_t *wr = (const uint32_t *)(slot + (16u * m + j) * (S::UPR * 16u));
                    uint32_t c0, c1;
                    if constexpr (Q51) {
                        const uint32_t *blk = wr + 6u * s;
                        const uint32_t dm = blk[0], hbits = (blk[1] >> (8u * g)) & 0xffu;
                        const uint2 qv = *(const uint2 *)(blk + 2u + 2u * (g & 1u));
                        c0 = ((qv.x >> shn) & 0x0f0f0f0fu) | spread4(hbits & 15u);
                        c1 = ((qv.y >> shn) & 0x0f0f0f0fu) | spread4(hbits >> 4);
                        d[m] = half_bits(dm) * 0x1p-5f;
                        mins[m][s] = dm >> 16;
                        check(dm);
                    } else if (s % 2u == 0u) {
                        /* block s at byte 34 s, codes of k-group g at + 2 + 8 g */
                        const uint32_t *blk = wr + 17u * (s / 2u);
                        d[m] = half_bits(blk[0]);
                        check(blk[0] & 0xffffu);
                        const uint32_t q0 = blk[2u * g], q1 = blk[2u * g + 1u], q2 = blk[2u * g + 2u];
                        c0 = kq_align2(q1, q0, 2u) ^ 0x80808080u;
                        c1 = kq_align2(q2, q1, 2u) ^ 0x80808080u;
                    } else {
                        const uint32_t *blk = wr + (34u * s - 2u) / 4u;
                        d[m] = half_bits(blk[0] >> 16);
                        check(blk[0] >> 16);
                        c0 = blk[1u + 2u * g] ^ 0x80808080u;
                        c1 = blk[2u + 2u * g] ^ 0x80808080u;
                    }
                    b[m] = cat(bytes_lo(c0) + bias, bytes_hi(c0) + bias, bytes_lo(c1) + bias,
                               bytes_hi(c1) + bias);
                }
            };
            read(0u);
            read(1u);
#pragma unroll
            for (uint32_t s = 0; s < 4u; ++s) {
                f4 t[NT][NF];
                decode(s);
#pragma unroll
                for (uint32_t i = 2u * NF * s; i < 2u * NF * (s + 1u); ++i) {
                    const uint32_t f = i % NF;
                    const bool lo_half = i / NF % 2u != 0u;
                    if (i + 2u < 8u * NF) read(i + 2u);
#pragma unroll
                    for (uint32_t m = 0; m < NT; ++m)
                        t[m][f] = mfma32(x[i % 3u], b[m], lo_half ? t[m][f] : zero);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
                }
#pragma unroll
                for (uint32_t f = 0; f < NF; ++f)
#pragma unroll
                    for (uint32_t m = 0; m < NT; ++m)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[m][f][e] = fmaf(d[m], t[m][f][e], acc[m][f][e]);
            }
            if constexpr (Q51) {
                /* k-group 0 the sums' hi halves, 1 the lo halves */
                const uint32_t on = 0u - (uint32_t)(g < 2u);
                const uint8_t *p = msum + par * S::MINS + (c_step * kM + j) * 16u + 8u * (g & 1u);
#pragma unroll
                for (uint32_t m = 0; m < NT; ++m) {
                    const h4 mn = __builtin_bit_cast(h4, make_uint2((mins[m][0] | (mins[m][1] << 16)) & on,
                                                                    (mins[m][2] | (mins[m][3] << 16)) & on));
#pragma unroll
                    for (uint32_t f = 0; f < NF; ++f)
                        acc[m][f] = mfma16(*(const h4 *)(p + 256u * f), mn, acc[m][f]);
                }
            }
        }
    };
    /* the finished tile: token i = 16 f + 4 g + q, row of this lane */
    auto store = [&](bool add) {
        const bool sh = (cur.ex & kShared) != 0u;
        const uint32_t pos0 = sh && !a.plain ? a.pairs + cur.first : cur.first;
        const uint32_t col = sh && a.plain ? a.rows : 0u;
#pragma unroll
        for (uint32_t f = 0; f < 4u; ++f) {
            if (16u * f >= cur.count) break;
#pragma unroll
            for (uint32_t q = 0; q < 4u; ++q) {
                const uint32_t i = 16u * f + 4u * g + q;
                const int sg = s_sig[par * kM + i];
                float *o = a.out + (size_t)(pos0 + i) * a.stride + col;
                if constexpr (GU) {
                    const uint32_t row = c_tile * TROWS + 16u * w + j;
                    const bool valid = i < cur.count && row < a.rows;
                    const float gv = ldexpf(acc[0][f][q], -sg), uv = ldexpf(acc[1][f][q], -sg);
                    /* silu(g) u with the hardware exponential, as the
                     * 16-token pass */
                    const float v = gv * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-gv * 1.44269504088896341f)) * uv;
                    bad |= valid && (!kq_isfinite(gv) || !kq_isfinite(uv) || !kq_isfinite(v));
                    if (valid) o[row] = v;
                } else {
#pragma unroll
                    for (uint32_t m = 0; m < NT; ++m) {
                        const uint32_t row = c_tile * TROWS + 16u * NT * w + 16u * m + j;
                        const bool valid = i < cur.count && row < a.rows;
                        float v = ldexpf(acc[m][f][q], (S::MINS != 0u ? 5 : 0) - sg);
                        if (add && valid) v += o[row];
                        bad |= valid && !kq_isfinite(v);
                        if (valid) o[row] = v;
                    }
                }
            }
        }
    };

    request(0u);
    const uint32_t n = (hi - lo + peers - 1u) / peers * steps;
    for (uint32_t k = 0; k < n; ++k) {
        /* step k's loads of this wave, then of every wave, have landed; the
         * other buffer's readers are done */
        wait_vm_all();
        kq_lds_barrier();
        if constexpr (S::K) {
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                hd[m] = arrived(nhd[m], turn);
                qa[m] = arrived(nqa[m], turn);
                qb[m] = arrived(nqb[m], turn);
                if constexpr (Q5) qh[m] = arrived(nqh[m], turn);
            }
        }
        if (k + 1u < n) request((k + 1u) & 1u);
        const uint8_t *img = lds + (k & 1u) * S::IMG;
        const uint8_t *slot = slots + ((k & 1u) * NW + w) * S::SLOT;
        switch ((cur.count + 15u) / 16u) {
        case 1u: product(std::integral_constant<uint32_t, 1u>{}, img, slot); break;
        case 2u: product(std::integral_constant<uint32_t, 2u>{}, img, slot); break;
        case 3u: product(std::integral_constant<uint32_t, 3u>{}, img, slot); break;
        default: product(std::integral_constant<uint32_t, 4u>{}, img, slot); break;
        }
        ++c_step;
        if constexpr (!GU) {
            if (++c_run == kRun && c_step != steps) {
                store(c_step != kRun);
                clear();
                c_run = 0u;
            }
        }
        if (c_step == steps) {
            store(!GU && steps > kRun);
            clear();
            c_step = 0u;
            c_run = 0u;
            c_t += peers;
            c_tile += peers;
            if (c_tile >= nt && k + 1u < n) {
                const uint32_t it = c_t / nt;
                c_tile = c_t - it * nt;
                cur = item(it);
                par ^= 1u;
            }
        }
    }
    /* (merged into the K formats' flag it cost the Q5_K pass 34 spilled
     * registers: 638 against 581 us at 2000 tokens) */
    if constexpr (!S::K) malformed = !(finite.x == finite.x) || !(finite.y == finite.y);
    if (malformed) kq_flag(a.status, KQ_DEV_MALFORMED);
    if (bad) kq_flag(a.status, KQ_DEV_NUMERIC);
}

template <uint32_t FMT, bool GU, uint32_t NW, uint32_t NT>
hipError_t launch(const GmArgs &a, hipStream_t s) {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0, n = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e == hipSuccess)
            e = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess || n <= 0) return e != hipSuccess ? e : hipErrorInvalidValue;
        cus = n;
    }
    hipLaunchKernelGGL((gm_product<FMT, GU, NW, NT>), dim3(((uint32_t)cus + kDies - 1u) / kDies * kDies), dim3(NW * 64u), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_plain_type(uint32_t type, const GmArgs &a, hipStream_t s) {
    switch (type) {
    case KQ_LAUNCH_Q5_1: return launch<KQ_LAUNCH_Q5_1, false, 8u, 2u>(a, s);
    case KQ_LAUNCH_Q6_K: return launch<KQ_LAUNCH_Q6_K, false, 8u, 2u>(a, s);
    case KQ_LAUNCH_Q8_0: return launch<KQ_LAUNCH_Q8_0, false, 8u, 2u>(a, s);
    default: return hipErrorInvalidValue;
    }
}

/* offsets are 31 bits; kOut stays past every buffer for each step's addition */
bool fits(uint64_t rows, uint64_t row_bytes, uint64_t src_rows, uint64_t k) {
    return rows * row_bytes < (UINT64_C(1) << 31) && src_rows * k * 2u < (UINT64_C(1) << 31);
}

}  // namespace

extern "C" int kq_launch_gm_gate_up_supported(uint32_t type, uint32_t rows, uint32_t k,
                                              uint32_t tokens) {
    return is_k(type) && k != 0u && k % 256u == 0u &&
           fits(rows, k / 256u * (uint64_t)unit_bytes(type), tokens, k);
}

extern "C" int kq_launch_gm_matrix_supported(uint32_t type, uint32_t rows, uint32_t k,
                                             uint32_t src_rows) {
    const bool k_ok = type == KQ_LAUNCH_Q8_0   ? k % 128u == 0u
                      : type == KQ_LAUNCH_Q5_1 ? k % 128u == 0u && k <= 1024u
                      : type == KQ_LAUNCH_Q6_K ? k % 512u == 0u /* rows of whole dwords */
                                               : false;
    return k_ok && k != 0u && fits(rows, k / 128u * (uint64_t)unit_bytes(type) / 2u, src_rows, k);
}

extern "C" hipError_t kq_launch_gm_gate_up(uint32_t type, const void *gate, const void *up,
                                           const void *shared_gate, const void *shared_up,
                                           uint32_t rows, uint32_t k, const void *staged,
                                           uint32_t tokens, uint32_t top_k,
                                           const uint32_t *perm_tok, const void *items,
                                           float *act, uint32_t *status, hipStream_t s) {
    if (!kq_launch_gm_gate_up_supported(type, rows, k, tokens)) return hipErrorInvalidValue;
    const kq::StagedX sx = kq::staged_at(const_cast<void *>(staged), tokens, k);
    GmArgs a = {};
    a.w0 = (const uint8_t *)gate;
    a.w1 = (const uint8_t *)up;
    a.s0 = (const uint8_t *)shared_gate;
    a.s1 = (const uint8_t *)shared_up;
    a.xh = sx.xh;
    a.xl = sx.xl;
    a.sx = sx.sx;
    a.sig = sx.sig;
    a.perm_tok = perm_tok;
    a.n_items = (const uint32_t *)items;
    a.items = (const uint32_t *)items + 4;
    a.src_rows = tokens;
    a.pairs = tokens * top_k;
    a.rows = a.stride = rows;
    a.k = k;
    a.out = act;
    a.status = status;
    return type == KQ_LAUNCH_Q5_K ? launch<KQ_LAUNCH_Q5_K, true, 8u, 2u>(a, s)
                                  : launch<KQ_LAUNCH_Q4_K, true, 8u, 2u>(a, s);
}

extern "C" hipError_t kq_launch_gm_down(uint32_t type, const void *down, const void *shared_down,
                                        uint32_t rows, uint32_t k, const void *xh, const void *xl,
                                        const int *sig, uint32_t tokens, uint32_t top_k,
                                        const void *items, float *out, uint32_t *status,
                                        hipStream_t s) {
    GmArgs a = {};
    a.src_rows = tokens * top_k + tokens;
    if (!kq_launch_gm_matrix_supported(type, rows, k, a.src_rows)) return hipErrorInvalidValue;
    a.w0 = (const uint8_t *)down;
    a.s0 = (const uint8_t *)shared_down;
    a.xh = (const _Float16 *)xh;
    a.xl = (const _Float16 *)xl;
    a.sig = sig;
    a.n_items = (const uint32_t *)items;
    a.items = (const uint32_t *)items + 4;
    a.pairs = tokens * top_k;
    a.rows = a.stride = rows;
    a.k = k;
    a.out = out;
    a.status = status;
    return launch_plain_type(type, a, s);
}

extern "C" hipError_t kq_launch_gm_dense(uint32_t type, const void *w0, const void *w1,
                                         uint32_t rows, uint32_t k, const void *xh, const void *xl,
                                         const int *sig, uint32_t tokens, float *out,
                                         uint32_t *status, hipStream_t s) {
    if (!kq_launch_gm_matrix_supported(type, rows, k, tokens)) return hipErrorInvalidValue;
    GmArgs a = {};
    a.w0 = (const uint8_t *)w0;
    a.s0 = (const uint8_t *)w1;
    a.xh = (const _Float16 *)xh;
    a.xl = (const _Float16 *)xl;
    a.sig = sig;
    a.src_rows = tokens;
    a.rows = rows;
    a.k = k;
    a.plain = w1 != nullptr ? 2u : 1u;
    a.stride = a.plain * rows;
    a.out = out;
    a.status = status;
    return launch_plain_type(type, a, s);
}
