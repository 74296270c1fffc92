/*
 * kq_mfma.h — GGUF blocks as matrix-core operands: the pieces that the
 * matrix-core products share. Codes enter fp16 exactly; a step's k order is
 * the one that lets a lane read its bytes in one piece.
 */
#ifndef KQ_MFMA_H
#define KQ_MFMA_H

#include "kq_device.h"
#include "kq_launch.h"

namespace kq {
namespace mf {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kUnit = 256; /* columns per unit */

__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
/* bytes 0, 1 / 2, 3 of m as fp16 1024 + byte */
__device__ __forceinline__ h2 bytes_lo(uint32_t m) {
    return as_h2(__builtin_amdgcn_perm(0x64646464u, m, 0x04010400u));
}
__device__ __forceinline__ h2 bytes_hi(uint32_t m) {
    return as_h2(__builtin_amdgcn_perm(0x64646464u, m, 0x04030402u));
}
/* and as the subnormals byte 2^-24 */
__device__ __forceinline__ h2 tiny_lo(uint32_t m) {
    return as_h2(__builtin_amdgcn_perm(0u, m, 0x04010400u));
}
__device__ __forceinline__ h2 tiny_hi(uint32_t m) {
    return as_h2(__builtin_amdgcn_perm(0u, m, 0x04030402u));
}
__device__ __forceinline__ h2 fma2(h2 a, h2 b, h2 c) { return __builtin_elementwise_fma(a, b, c); }
__device__ __forceinline__ h2 splat(float v) { return h2{(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ h8 cat(h2 a, h2 b, h2 c, h2 d) {
    return h8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}
__device__ __forceinline__ float half_bits(uint32_t h) { return kq_f16_to_f32_hw(h); }
/* bits 0..3 of x (x < 16) to bit 4 of bytes 0..3 */
__device__ __forceinline__ uint32_t spread4(uint32_t x) {
    return (kq_mul_u24(x, 0x00204081u) & 0x01010101u) << 4;
}
__device__ __forceinline__ f4 mfma32(h8 a, h8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma16(h4 a, h4 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
}

constexpr bool is_k(uint32_t f) { return f == KQ_LAUNCH_Q4_K || f == KQ_LAUNCH_Q5_K; }

/* bytes of 256 columns */
constexpr uint32_t unit_bytes(uint32_t f) {
    return f == KQ_LAUNCH_Q4_K ? 144u
           : f == KQ_LAUNCH_Q5_K ? 176u
           : f == KQ_LAUNCH_Q6_K ? 210u
           : f == KQ_LAUNCH_Q8_0 ? 272u
           : f == KQ_LAUNCH_Q5_1 ? 192u
           : f == KQ_LAUNCH_IQ4_NL ? 144u : 0u;
}
/* columns per block */
constexpr uint32_t block_cols(uint32_t f) {
    return is_k(f) || f == KQ_LAUNCH_Q6_K ? 256u : 32u;
}

/* the middle of the K formats' codes */
constexpr float k_mid(uint32_t f) { return f == KQ_LAUNCH_Q5_K ? 16.0f : 8.0f; }

/* scale-like six-bit fields 4 h .. 4 h + 3 of a block's mins, one per byte */
__device__ __forceinline__ uint32_t k_mins(const uint4 hd, uint32_t h) {
    const uint32_t k0 = 0u - (uint32_t)(h == 0u);
    return ((hd.z & 0x3f3f3f3fu) & k0) |
           ((((hd.w >> 4) & 0x0f0f0f0fu) | ((hd.z >> 2) & 0x30303030u)) & ~k0);
}
__device__ __forceinline__ uint32_t k_scales(const uint4 hd, uint32_t h) {
    const uint32_t k0 = 0u - (uint32_t)(h == 0u);
    return ((hd.y & 0x3f3f3f3fu) & k0) |
           (((hd.w & 0x0f0f0f0fu) | ((hd.y >> 2) & 0x30303030u)) & ~k0);
}
/* the scales of the sub-blocks that have a min, 0 of the others */
__device__ __forceinline__ uint32_t k_centres(const uint4 hd, uint32_t h) {
    const uint32_t some = ((k_mins(hd, h) + 0x7f7f7f7fu) & 0x80808080u) >> 7;
    return k_scales(hd, h) & ((some << 8) - some);
}

/* The scales of sub-blocks 2 pair and 2 pair + 1 of a Q4_K or Q5_K block, the
 * low and the high nibbles of bytes 32 pair .. + 31. A code byte under a zero
 * high byte is the subnormal q 2^-24 (16 q for Q4_K's high nibbles, left in
 * place); one fused multiply-add makes it (q - c) s 2^-14: exact. CENTRED: c
 * is the middle of the codes' range (at most 1008 2^-14), their mean stays out
 * of the long sums and c s comes back beside the mins (k_centres); otherwise,
 * and in sub-blocks without a min, whose zero codes are zero weights, c is 0
 * (at most 1953 2^-14). */
template <uint32_t FMT, bool CENTRED>
struct KPair {
    h2 S[2], C[2];

    __device__ __forceinline__ KPair(const uint4 hd, uint32_t pair) {
        constexpr float c = CENTRED ? k_mid(FMT) * -0x1p-14f : 0.0f;
        uint32_t s0, s1, m0, m1;
        kq_k_scale_pair(pair, hd.y, hd.z, hd.w, &s0, &m0, &s1, &m1);
        S[0] = splat((float)s0 * 1024.0f);
        S[1] = splat((float)s1 * (FMT == KQ_LAUNCH_Q5_K ? 1024.0f : 64.0f));
        C[0] = splat(CENTRED && m0 != 0u ? (float)s0 * c : 0.0f);
        C[1] = splat(CENTRED && m1 != 0u ? (float)s1 * c : 0.0f);
    }
    /* the weights of eight columns of sub-block 2 pair + high: r0, r1 their
     * qs bytes, h0, h1 their qh bytes (Q5_K) */
    __device__ __forceinline__ h8 weights(uint32_t high, uint32_t pair, uint32_t r0, uint32_t r1,
                                          uint32_t h0, uint32_t h1) const {
        uint32_t m0, m1;
        if constexpr (FMT == KQ_LAUNCH_Q5_K) {
            const uint32_t sh = 2u * pair + high;
            m0 = ((high ? r0 >> 4 : r0) & 0x0f0f0f0fu) | (((h0 >> sh) & 0x01010101u) << 4);
            m1 = ((high ? r1 >> 4 : r1) & 0x0f0f0f0fu) | (((h1 >> sh) & 0x01010101u) << 4);
        } else {
            m0 = high ? kq_and_f0(r0) : kq_and_0f(r0);
            m1 = high ? kq_and_f0(r1) : kq_and_0f(r1);
        }
        return cat(fma2(tiny_lo(m0), S[high], C[high]), fma2(tiny_hi(m0), S[high], C[high]),
                   fma2(tiny_lo(m1), S[high], C[high]), fma2(tiny_hi(m1), S[high], C[high]));
    }
};

/* four bytes as halves */
__device__ __forceinline__ h4 byte_halves(uint32_t q) {
    const h2 a = bytes_lo(q) + splat(-1024.0f), b = bytes_hi(q) + splat(-1024.0f);
    return h4{a.x, a.y, b.x, b.y};
}

/* dword 2 i + h of 32 bytes */
__device__ __forceinline__ uint32_t dword_of(const uint4 &a, const uint4 &b, uint32_t i, uint32_t h) {
    const uint4 &q = (i & 2u) ? b : a;
    return (i & 1u) ? (h ? q.w : q.z) : (h ? q.y : q.x);
}

}  // namespace mf
}  // namespace kq

#endif
