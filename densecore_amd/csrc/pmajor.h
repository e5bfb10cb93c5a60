// The "P-major" activation layout that the matrix-core GEMMs and the kernels for nine to 64 rows read: sixteen activation
// rows x one super-block per tile of 4688 bytes, written by quantize_q8k_pmajor_kernel (prefill.hip), tile (b, mt) at
// (b * m_tiles + mt) * 4688.
//   [j 0..3][kq 0..3][tok 0..15][16 B]   codes: bytes 0..7 = sub-block ga(j), elements 8kq..8kq+7,
//                                        bytes 8..15 = sub-block gb(j), same elements, with
//                                        (ga, gb) = (0,2) (1,3) (4,6) (5,7) for j = 0..3 -- the pairs
//                                        that one 16-byte word of a weight tile holds per nibble half
//   [tok][32 B] at 4096                  fp16 base-128 digits of the sub-block code sums: l_0..l_7, then 128 h_0..128 h_7
//   [tok] fp32 at 4608                   block scale d
//   16 zero bytes at 4672                what the lanes of k-groups 2 and 3 feed a K = 32 min MFMA
//
// The same of one row x one super-block in 320 bytes ("row layout", for rows that are gathered into tiles; row m of n rows and
// super-block b at (b * n + m) * 320): the codes [j][kq][16 B], the sixteen digits at 256, the scale at 288.
#pragma once

#include "common.h"

namespace mq {

constexpr int kPTileBytes = 4688;
constexpr int kPTileWords = kPTileBytes / 16;  // 293
constexpr int kPDigitOff = 4096, kPScaleOff = 4608, kPZeroOff = 4672;
constexpr int kPRowBytes = 320, kPRowDigitOff = 256, kPRowScaleOff = 288;

#if defined(__HIPCC__)
typedef unsigned short v2us __attribute__((ext_vector_type(2)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

// four bytes (each <= 15) times a 3-bit digit, bytewise: two 16-bit products whose bytes do not carry into each
// other (15 * 7 < 256).  The digit is half H of `digits`, taken for both products (the operand-select bits of the
// packed multiply: no instruction of its own).
template <int H>
__device__ __forceinline__ uint32_t scale_bytes(uint32_t nibbles, uint32_t digits) {
    const v2us a = __builtin_bit_cast(v2us, nibbles);
    const v2us d = __builtin_bit_cast(v2us, digits);
    const v2us dd = H ? v2us{d.y, d.y} : v2us{d.x, d.x};
    return __builtin_bit_cast(uint32_t, (v2us)(a * dd));
}

// bytes i and i + 1 of `word` as two 16-bit numbers (one v_perm_b32: selector 0x0c yields a zero byte)
__device__ __forceinline__ uint32_t digit_pair(uint32_t word, int i) {
    return __builtin_amdgcn_perm(0u, word, 0x0c000c00u | (uint32_t)i | ((uint32_t)(i + 1) << 16));
}

// the eight 6-bit mins of a Q4_K / Q5_K block (bytes of two words) as fp16: 0x6400 | n is 1024 + n, two at a time
__device__ __forceinline__ v8h mins_to_half(uint32_t mn03, uint32_t mn47) {
    const v2h bias = {(_Float16)1024.0f, (_Float16)1024.0f};
    const v2h m01 = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64006400u, mn03, 0x05010500u)) - bias;
    const v2h m23 = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64006400u, mn03, 0x05030502u)) - bias;
    const v2h m45 = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64006400u, mn47, 0x05010500u)) - bias;
    const v2h m67 = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64006400u, mn47, 0x05030502u)) - bias;
    return v8h{m01.x, m01.y, m23.x, m23.y, m45.x, m45.y, m67.x, m67.y};
}

// The four wavefronts of a workgroup request activation tiles (copy_words 16-byte words, contiguous in HBM) straight into LDS
// (lds_direct, common.h): a run of 64-word requests is a linear copy that never touches a register.  The requests fill the buffer that
// is not being read; the kernel waits for them, with vmcnt(0) and a barrier, before it is.
__device__ __forceinline__ void request_a_tiles(const uint8_t* __restrict__ src, uint8_t* buf, int copy_words, int wave,
                                                int lane) {
    // The address is a scalar base and the lane's 16 l: 22 registers less than an address per lane and request, which the compiler kept
    // over the whole loop.
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_ptr_t)buf;
    const uint32_t lane_off = (uint32_t)lane * 16u;
    const int full = copy_words >> 6;  // whole requests; everything but the lane's offset is scalar work
    const uint8_t* g = src + (size_t)wave * 1024;
    uint32_t dst = lds_base + (uint32_t)wave * 1024u;
    for (int q = wave; q < full; q += 4, g += 4096, dst += 4096)
        lds_direct<16>(g, lane_off, dst);
    if ((full & 3) == wave && lane < (copy_words & 63))  // the rest of the last tile, at the request behind this wavefront's last one
        lds_direct<16>(g, lane_off, dst);
}
#endif

}  // namespace mq
