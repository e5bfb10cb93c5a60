// Q4_K, Q5_K and Q6_K weight tiles expanded to the byte operands of two int8 MFMA chains (the matrix-core GEMM and the kernels
// for nine to 64 rows).
#pragma once

#include "decode_tile.h"
#include "pmajor.h"

namespace mq {

#if defined(__HIPCC__)
// A weight tile of 16 rows x one super-block as the B operands of the MFMA chains: weight integer = (hi << kDigitShift) + lo,
// both signed bytes, so that two chains of four K = 64 MFMAs form the whole super-block's integer whatever the type.
//   Q4_K  scale * code <= 945: hi = s1 * code, lo = s0 * code for scale = 8 s1 + s0 (both <= 105, formed bytewise: three and a
//         half vector instructions per four weights)
//   Q5_K  scale * code <= 1953, Q6_K  4 * scale * (code - 32) in +-16384 (the tile holds 4 (code - 32), see common.h; the
//         factor is taken out of d): the product is formed in 16 bits and cut into a high byte and a SIGNED low byte,
//         t = scale * code + 128, hi = t >> 8, lo = (t & 255) - 128
// The digits of 16-bit products replace a third chain for the fifth code bit (Q5_K: thirteen MFMAs per tile and super-block ->
// nine) and five chains over digits of both factors (Q6_K: twenty -> eight): the launch is bound by MFMA and vector issue at the
// card's power limit, so that is what it gains: 14336 x 4096 at 512 / 2048 rows Q5_K 108 / 391 -> 87 / 297, Q6_K 149 / 541 -> 84 / 286 us.
// Sixteen-bit products cost ten and a half vector instructions per four weights, the fifth bits as a chain of their own three
// less but four MFMAs and four shift-adds per activation tile more: kernels of one and two activation tiles per weight tile
// keep the third chain for Q5_K (FFN of 4096 -> 14336 -> 4096 at 30 rows 47.5 us, 48.0 with the digits).
struct WTile {
    v4i hi[4], lo[4];  // B operands of the four chunk pairs
    v4i b5[4];         // third chain only: the fifth code bits times the whole 6-bit scale, weight += 16 * b5
    v8h mins;          // Q4_K, Q5_K: B operand of the min MFMA: the eight mins as fp16, in every k-group
    float d, dmin;     // (Q6_K: d / 4, no dmin)
};
template <int WT, int MT>
constexpr bool kFifthChain = WT == kWtQ5 && MT <= 2;
template <int WT, int MT>
constexpr int kDigitShift = WT == kWtQ4 || kFifthChain<WT, MT> ? 3 : 8;
// the integer sums of the chains combined (b5: zeros without a third chain)
template <int WT, int MT>
__device__ __forceinline__ int join_digits(int hi, int lo, int b5) {
    const int dot = (hi << kDigitShift<WT, MT>) + lo;
    return kFifthChain<WT, MT> ? dot + (b5 << 4) : dot;
}

// Four products a[i] * s + 128 of code bytes (`even`, `odd`: codes 0, 2 and 1, 3 of a word as 16-bit numbers) and the 16-bit
// scale in half H of `scale`, cut into high bytes and signed low bytes in the order of the codes.
template <int H>
__device__ __forceinline__ void scale_digits(uint32_t even, uint32_t odd, uint32_t scale, int& hi, int& lo) {
    const v2us s = __builtin_bit_cast(v2us, scale);
    const v2us ss = H ? v2us{s.y, s.y} : v2us{s.x, s.x}, bias = {128, 128};
    const uint32_t te = __builtin_bit_cast(uint32_t, (v2us)(__builtin_bit_cast(v2us, even) * ss + bias));
    const uint32_t to = __builtin_bit_cast(uint32_t, (v2us)(__builtin_bit_cast(v2us, odd) * ss + bias));
    hi = (int)__builtin_amdgcn_perm(to, te, 0x07030501u);
    lo = (int)(__builtin_amdgcn_perm(to, te, 0x06020400u) ^ 0x80808080u);
}

// Q5_K: the codes are nibble + 16 * bit (bit s of the bytes of qh = fifth bit in sub-block s, core/src/kernels/hwy/hwy_moe_quant.cc:177-200).
template <bool Q5, bool FIFTH>
__device__ __forceinline__ void expand_tile(const v4u seg0, const v4u seg1, const v4u hdr, const v2u qh, int kq, WTile& t) {
    // 6-bit scales and mins (core/src/kernels/hwy/hwy_moe_quant.cc:90-101), four to a word
    const uint32_t sc03 = hdr.y & 0x3f3f3f3fu, mn03 = hdr.z & 0x3f3f3f3fu;
    const uint32_t sc47 = (hdr.w & 0x0f0f0f0fu) | (((hdr.y >> 6) & 0x03030303u) << 4);
    const uint32_t mn47 = ((hdr.w >> 4) & 0x0f0f0f0fu) | (((hdr.z >> 6) & 0x03030303u) << 4);
    const v4u seg[2] = {seg0, seg1};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        // (the digits ahead of the codes: formed behind them, the GEMM's schedule is 0.4 % slower -- gate/up pair of 14336 x 4096 at
        // 2048 rows 510.8 against 508.5 us)
        const uint32_t scw = i ? sc47 : sc03, s1w = (scw >> 3) & 0x07070707u, s0w = scw & 0x07070707u;
        // sub-blocks 4i .. 4i+3 are bytes 0..3 of the scale word
        const uint32_t l0 = seg[i].x & 0x0f0f0f0fu, l1 = seg[i].y & 0x0f0f0f0fu;  // sub-block 4i
        const uint32_t l2 = seg[i].z & 0x0f0f0f0fu, l3 = seg[i].w & 0x0f0f0f0fu;  // sub-block 4i+2
        const uint32_t h0 = (seg[i].x >> 4) & 0x0f0f0f0fu, h1 = (seg[i].y >> 4) & 0x0f0f0f0fu;  // 4i+1
        const uint32_t h2 = (seg[i].z >> 4) & 0x0f0f0f0fu, h3 = (seg[i].w >> 4) & 0x0f0f0f0fu;  // 4i+3
        if constexpr (Q5 && !FIFTH) {
            // scales of sub-blocks (4i, 4i+1) and (4i+2, 4i+3), two to a word
            const uint32_t abs_ = digit_pair(scw, 0), ces = digit_pair(scw, 2);
            const uint32_t codes[8] = {l0 | fifth_bits(qh.x, 4 * i), l1 | fifth_bits(qh.y, 4 * i), l2 | fifth_bits(qh.x, 4 * i + 2), l3 | fifth_bits(qh.y, 4 * i + 2),
                                       h0 | fifth_bits(qh.x, 4 * i + 1), h1 | fifth_bits(qh.y, 4 * i + 1), h2 | fifth_bits(qh.x, 4 * i + 3), h3 | fifth_bits(qh.y, 4 * i + 3)};
            int hi[8], lo[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t even = codes[k] & 0x00ff00ffu, odd = __builtin_amdgcn_perm(0u, codes[k], 0x0c030c01u);
                const uint32_t sc = (k & 2) ? ces : abs_;
                if (k < 4) scale_digits<0>(even, odd, sc, hi[k], lo[k]);
                else scale_digits<1>(even, odd, sc, hi[k], lo[k]);
            }
            t.hi[2 * i] = v4i{hi[0], hi[1], hi[2], hi[3]}, t.lo[2 * i] = v4i{lo[0], lo[1], lo[2], lo[3]};
            t.hi[2 * i + 1] = v4i{hi[4], hi[5], hi[6], hi[7]}, t.lo[2 * i + 1] = v4i{lo[4], lo[5], lo[6], lo[7]};
        } else {
            // digits of sub-blocks (4i, 4i+1) and (4i+2, 4i+3), two to a word
            const uint32_t ab1 = digit_pair(s1w, 0), ab0 = digit_pair(s0w, 0);
            const uint32_t ce1 = digit_pair(s1w, 2), ce0 = digit_pair(s0w, 2);
            t.hi[2 * i] = v4i{(int)scale_bytes<0>(l0, ab1), (int)scale_bytes<0>(l1, ab1), (int)scale_bytes<0>(l2, ce1),
                              (int)scale_bytes<0>(l3, ce1)};
            t.lo[2 * i] = v4i{(int)scale_bytes<0>(l0, ab0), (int)scale_bytes<0>(l1, ab0), (int)scale_bytes<0>(l2, ce0),
                              (int)scale_bytes<0>(l3, ce0)};
            t.hi[2 * i + 1] = v4i{(int)scale_bytes<1>(h0, ab1), (int)scale_bytes<1>(h1, ab1), (int)scale_bytes<1>(h2, ce1),
                                  (int)scale_bytes<1>(h3, ce1)};
            t.lo[2 * i + 1] = v4i{(int)scale_bytes<1>(h0, ab0), (int)scale_bytes<1>(h1, ab0), (int)scale_bytes<1>(h2, ce0),
                                  (int)scale_bytes<1>(h3, ce0)};
            if constexpr (FIFTH) {  // scale * bit <= 63 is a byte
                const uint32_t abs_ = digit_pair(scw, 0), ces = digit_pair(scw, 2);  // whole scales of sub-blocks (4i, 4i+1), (4i+2, 4i+3)
                auto bits = [&](uint32_t word, int sb) { return (word >> sb) & 0x01010101u; };
                t.b5[2 * i] = v4i{(int)scale_bytes<0>(bits(qh.x, 4 * i), abs_), (int)scale_bytes<0>(bits(qh.y, 4 * i), abs_),
                                  (int)scale_bytes<0>(bits(qh.x, 4 * i + 2), ces), (int)scale_bytes<0>(bits(qh.y, 4 * i + 2), ces)};
                t.b5[2 * i + 1] = v4i{(int)scale_bytes<1>(bits(qh.x, 4 * i + 1), abs_), (int)scale_bytes<1>(bits(qh.y, 4 * i + 1), abs_),
                                      (int)scale_bytes<1>(bits(qh.x, 4 * i + 3), ces), (int)scale_bytes<1>(bits(qh.y, 4 * i + 3), ces)};
            }
        }
    }
    t.mins = mins_to_half(mn03, mn47);
    t.d = half_bits_to_float(hdr.x & 0xffffu);
    t.dmin = half_bits_to_float(hdr.x >> 16);
}

// Q6_K: weight = d * scale_g * (code - 32), sixteen signed 8-bit scales per super-block, one per 16 weights
// (core/src/llm/matmul/q6_small_batch.h:13-92).  Word jj = 2 j + zp of the tile keeps each 64-byte run of nibbles as two 32-weight
// sub-blocks (z = zp and zp + 2 of half j), the pairs the P-major layout puts side by side.
__device__ __forceinline__ void expand_tile6(const v4u ql0, const v4u ql1, const v4u qh, const v4u sc, uint32_t dw, int kq, WTile& t) {
    typedef short v2s __attribute__((ext_vector_type(2)));
    const uint32_t scw[4] = {sc.x, sc.y, sc.z, sc.w};
    const v4u qlw[2] = {ql0, ql1};
    const uint32_t qhw[4] = {qh.x, qh.y, qh.z, qh.w};
    // weights 128 j + 32 z + l, l = 8 kq .. 8 kq + 7, have scale 8 j + 2 z + (kq >> 1): byte 2 (z & 1) + (kq >> 1) of
    // scale word 2 j + (z >> 1); the scales of z = zp and zp + 2 as 16-bit numbers side by side
    const uint32_t pick0 = 0x040c000cu + (uint32_t)(kq >> 1) * 0x01000100u;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int zp = 0; zp < 2; ++zp) {
            const int jj = 2 * j + zp;
            const uint32_t raised = __builtin_amdgcn_perm(scw[2 * j + 1], scw[2 * j], pick0 + 0x02000200u * (uint32_t)zp);
            const uint32_t scale = __builtin_bit_cast(uint32_t, (v2s)(__builtin_bit_cast(v2s, raised) >> 8));
            const uint32_t src[2] = {zp ? qlw[j].z : qlw[j].x, zp ? qlw[j].w : qlw[j].y};
            int hi[4], lo[4];
#pragma unroll
            for (int h = 0; h < 2; ++h)        // h = 0: z = zp (low nibbles), h = 1: z = zp + 2 (high nibbles)
#pragma unroll
                for (int i = 0; i < 2; ++i) {  // the lane's eight weights of the sub-block, four to a word
                    const int z = zp + 2 * h, o = 2 * h + i;
                    const uint32_t nib = (h ? src[i] >> 2 : src[i] << 2) & 0x3c3c3c3cu;
                    const uint32_t top = qhw[2 * j + i];
                    const uint32_t b4 = ((z == 3 ? top : top << (6 - 2 * z)) & 0xc0c0c0c0u) | nib;  // 4 (code - 32) as signed bytes
                    const uint32_t even = __builtin_bit_cast(uint32_t, (v2s)(__builtin_bit_cast(v2s, b4 << 8) >> 8));
                    const uint32_t odd = __builtin_bit_cast(uint32_t, (v2s)(__builtin_bit_cast(v2s, b4) >> 8));
                    if (h == 0) scale_digits<0>(even, odd, scale, hi[o], lo[o]);
                    else scale_digits<1>(even, odd, scale, hi[o], lo[o]);
                }
            t.hi[jj] = v4i{hi[0], hi[1], hi[2], hi[3]};
            t.lo[jj] = v4i{lo[0], lo[1], lo[2], lo[3]};
        }
    t.d = __fmul_rn(half_bits_to_float(dw & 0xffffu), 0.25f);
}
#endif

}  // namespace mq
