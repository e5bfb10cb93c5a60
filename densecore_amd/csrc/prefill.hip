// Prefill GEMM for gfx950: C[M][N] = q8k(A[M][K]) . W_q4k[N][K]^T for M in the hundreds and above,
// where the work is arithmetic on the int8 matrix cores rather than weight streaming
// (RunQ4KRawBatchedDenseGemm, core/src/backend/cpu_backend_q4k_dense.cpp:57-101, behind
// CpuBackend::MatMulGgmlQuantizedTransB, core/src/backend/cpu_backend_quantized_matmul.cpp:150-175).
//
// The per-sub-block 6-bit scales are what keeps Q4_K off a plain int8 GEMM.  Here they are folded
// into the weight operand so that v_mfma_i32_16x16x64_i8 accumulates over the whole super-block:
//     scale = 8*s1 + s0  (two 3-bit digits)   ->   (s1*q4) and (s0*q4) both fit a signed byte (<= 105)
//     dot_scaled = 8 * sum_k (s1*q4)_k q8_k  +  sum_k (s0*q4)_k q8_k                  (exact, int32)
// and the min term runs on the matrix cores as well, from the sub-block sums of the codes
// bs_g = bsums[2g] + bsums[2g+1] = 128*h_g + l_g (h in [-32, 31], l in [0, 127]):
//     min_dot = sum_g min_g (128 h_g)  +  sum_g min_g l_g
// which is the reference's sum_j bsums[j] * min[j/2] (core/src/llm/matmul/kquant_batched_kernels.h:285-297).
// One v_mfma_f32_16x16x32_f16 forms it: the sixteen operands l_g, 128 h_g and the mins are integers of at most
// thirteen bits, exact as fp16; every product and every partial sum is an integer below 2^24, so the fp32 result
// is the integer min_dot itself -- the value (float)min_dot that the update needs, with nothing to combine or
// convert on the vector unit.
// Nine MFMAs per 16x16 output tile and super-block (Q5_K the same, Q6_K eight: weight_digits.h), no per-sub-block vector
// work; the fp32 update
//     acc += yd * (d * dot_scaled - dmin * min_dot)
// is done once per super-block, as every reference kernel does (three fp32 operations per output, five vector
// instructions with the digits' shift-add and one conversion; the reference's
// grouping (d*yd) * dot_scaled - (dmin*yd) * min_dot takes four, and the update is what the kernel's vector unit is
// busy with: 308 against 325 us at M = 2048; the two groupings differ in the last bits only).
//
//   grid      = (row_wgs, groups, splits) of the shape that choose_shape takes; workgroup = 4 wavefronts
//   workgroup = 128 or 64 weight rows x up to 128 activation rows (tiles_per_wg tiles) x all super-blocks or a run of them;
//               per super-block the activation rows (up to 37 KB in the P-major layout) are staged in LDS, double-buffered
//               and requested one super-block ahead with LDS-direct loads
//   wavefront = 2 weight tiles (32 rows; 64-row workgroups: 1) x the activation tiles; it reads its weight tiles
//               straight from HBM in MFMA lane order and expands them in registers
//
// The activations come in the P-major layout (pmajor.h).
#include <hip/hip_ext.h>

#include "common.h"
#include "kernels.h"
#include "decode_tile.h"
#include "pmajor.h"
#include "q8k_block.h"
#include "weight_digits.h"

namespace mq {

namespace {

constexpr int kMTilesPerGroup = 8;             // activation tiles (of 16 rows) per workgroup
constexpr int kMTilesSmall = 2;                // ... of an expert-grouped launch whose experts hold a dozen or two rows
constexpr int kMTilesMid = 4;                  // ... or three or four dozen

// request_a_tiles (pmajor.h) with an address per lane and request, unrolled: the same copies.  Scalar addresses take 1 to 4 % off the
// wide forms and the pairs (Q6_K 14336 x 4096 at 512 rows 83.4 -> 80.5 us, Q4_K FFN 4096 -> 14336 at 2048 rows 765 -> 759), but
// the loop around a request costs the forms that have registers to spare: 64-row workgroups of Q4_K and Q6_K 19.3 with this | 19.8 with scalar
// addresses (Q6_K 4096 x 4096 at 100 rows; unrolled scalar requests 20.3).  Q5_K's wide forms had gained as much (6152 x 4096 at 1000 rows 84.0 |
// 85.6), but with loops of their own for five to eight tiles this spills 6, 18, 38 and 61 registers: they take scalar addresses (81.2).
template <int MT>
__device__ __forceinline__ void request_a_tiles_by_lane(const uint8_t* __restrict__ src, uint8_t* buf, int copy_words, int wave, int lane) {
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_ptr_t)buf;
    constexpr int kRounds = (MT * kPTileWords + 255) / 256;  // 4 waves x 64 words a round: ten rounds for eight tiles of 293 words
#pragma unroll
    for (int j = 0; j < kRounds; ++j) {
        const int first = (j * 4 + wave) * 64;
        if (first + lane < copy_words) {
            const uint8_t* g = src + (size_t)(first + lane) * 16;
            const uint32_t dst = lds_base + (uint32_t)first * 16u;  // wave-uniform; lane l lands at dst + 16*l
            lds_direct<16>(g, dst);
        }
    }
}

// request_a_tiles (pmajor.h) for rows that lie in the row layout (kPRowBytes each): tile t of the workgroup's tiles is fetched by wavefront t & 3, lane
// (kq, r) = 16 kq + r of request j the sixteen bytes that the tile holds there, from row rows[16 t + r].  Offsets of a lane's rows
// inside a super-block's plane:
template <int MT>
struct GatherOffsets {
    static constexpr int kTiles = (MT + 3) / 4;  // tiles per wavefront
    uint32_t code[kTiles], digit[kTiles], scale[kTiles];
    __device__ __forceinline__ void load(const int32_t* __restrict__ rows, int tiles, int wave, int lane) {
#pragma unroll
        for (int i = 0; i < kTiles; ++i) {
            const int t = wave + 4 * i < tiles ? wave + 4 * i : 0;
            const int rc = rows[16 * t + (lane & 15)], rd = rows[16 * t + ((lane >> 1) & 15)];  // -1: padding, any row will do (its results go nowhere)
            const uint32_t c = (uint32_t)(rc < 0 ? 0 : rc) * kPRowBytes, d = (uint32_t)(rd < 0 ? 0 : rd) * kPRowBytes;
            code[i] = c + (uint32_t)(lane >> 4) * 16u;
            digit[i] = d + kPRowDigitOff + (uint32_t)(lane & 1) * 16u;
            scale[i] = c + kPRowScaleOff;
        }
    }
};
template <int MT>
__device__ __forceinline__ void request_a_rows(const GatherOffsets<MT>& off, const uint8_t* __restrict__ plane, uint8_t* buf, int tiles, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < GatherOffsets<MT>::kTiles; ++i) {
        const int t = wave + 4 * i;
        if (t >= tiles) break;  // wave-uniform
        const uint32_t dst = (uint32_t)(uintptr_t)(lds_ptr_t)buf + (uint32_t)t * kPTileBytes;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            lds_direct<16>(plane + j * 64, off.code[i], dst + j * 1024);
        if (lane < 32) lds_direct<16>(plane, off.digit[i], dst + kPDigitOff);
        if (lane < 16) lds_direct<4>(plane, off.scale[i], dst + kPScaleOff);
    }
}

// kWTilesPerWave = 2: the 128 x 128 workgroup tile above.  1: 64 weight rows per workgroup, for launches whose
// 128-row workgroups would leave compute units without their two workgroups (M up to a few hundred).
// PAIR (two weight tiles per wavefront): the wavefront's two tiles are the SAME row tile of two matrices, gate
// (w) and up (w2), and what is stored is silu(gate) * up -- the two fp32 planes a gate launch and an up launch would
// write, and the pass that reads them back to form the product, never exist (for 2048 rows of a 4096 -> 14336 FFN that
// is 235 MB written and read).  The same accumulators, the same SiLU function on the same values: the same bits.
// MT: activation tiles (of 16 rows) a workgroup multiplies.  Eight for the dense product; the expert-grouped one also
// comes with two (items of 32 rows): with a dozen or two routed rows per expert a workgroup has one or two tiles, its
// accumulators for eight only cost registers and LDS -- and how many workgroups a compute unit holds is what hides the
// latency of a workgroup that walks eight super-blocks with a barrier each.
template <int kWTilesPerWave, int WT = kWtQ4, bool PAIR = false, int MT = kMTilesPerGroup, bool GATHER = false, bool kDense = false>
__global__ void __launch_bounds__(256, PAIR && MT == kMTilesMid && WT != kWtQ5 ? 3 : 2) prefill_gemm_kernel(const uint8_t* __restrict__ w, int64_t rowtiles, int64_t rows,
                                                           int64_t nb, const uint8_t* __restrict__ ap, int64_t m_tiles,
                                                           int64_t n_tokens, float* __restrict__ y, int64_t ldy, int sb_split,
                                                           int64_t split_stride, const int32_t* __restrict__ plan,
                                                           int64_t expert_bytes, const int32_t* __restrict__ out_rows,
                                                           const uint8_t* __restrict__ w_shared,
                                                           const uint8_t* __restrict__ w2 = nullptr,
                                                           const uint8_t* __restrict__ w2_shared = nullptr, int silu_mode = 0,
                                                           int tiles_per_wg = MT, const int32_t* __restrict__ a_rows = nullptr,
                                                           size_t a_plane = 0) {
    static_assert(!PAIR || kWTilesPerWave == 2, "the pair form is the two-tile kernel");
    extern __shared__ __align__(16) uint8_t a_lds[];  // two buffers of MT * kPTileBytes bytes
    constexpr int kBufBytes = MT * kPTileBytes;
    constexpr bool Q5 = WT == kWtQ5, Q6 = WT == kWtQ6;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kq = lane >> 4;
    // Dense: workgroup column blockIdx.y takes the next tiles_per_wg (<= MT) activation tiles.  Expert-grouped (plan != null):
    // it takes item blockIdx.y of the plan -- an expert's weights and a run of up to eight tiles of that expert's rows.
    int64_t mt0 = (int64_t)blockIdx.y * tiles_per_wg;
    int mt_count = (int)(m_tiles - mt0 < tiles_per_wg ? m_tiles - mt0 : tiles_per_wg);
    if (plan) {
        const int item = blockIdx.y;
        if (item >= plan[0]) return;  // the whole workgroup, before any barrier
        const int expert = plan[4 + 3 * item];  // -1: the shared expert's rows
        w = expert < 0 ? w_shared : w + (size_t)expert * (size_t)expert_bytes;
        if constexpr (PAIR) {
            w2 = expert < 0 ? w2_shared : w2 + (size_t)expert * (size_t)expert_bytes;
            if (expert < 0) silu_mode = plan[3];  // the shared expert's rows: its own SiLU form
        }
        mt0 = plan[5 + 3 * item];
        mt_count = plan[6 + 3 * item];
    }
    const int64_t rt0 = ((int64_t)blockIdx.x * 4 + wave) * (PAIR ? 1 : kWTilesPerWave);
    // weight tiles past the end are replaced by the last valid one and simply not stored
    int64_t rt[kWTilesPerWave];
#pragma unroll
    for (int t = 0; t < kWTilesPerWave; ++t) rt[t] = rt0 + (PAIR ? 0 : t) < rowtiles ? rt0 + (PAIR ? 0 : t) : rowtiles - 1;

    float acc[kWTilesPerWave][MT][4];
#pragma unroll
    for (int t = 0; t < kWTilesPerWave; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[t][m][i] = 0.0f;

    const int copy_words = mt_count * kPTileWords;
    // this lane's operand of the min MFMA: k-group 0 reads the l digits of token r, k-group 1 its 128 h digits, the others zeros
    const int digit_off = kq < 2 ? kPDigitOff + r * 32 + kq * 16 : kPZeroOff;
    const uint8_t* a_src = GATHER ? ap : ap + (size_t)mt0 * kPTileBytes;  // + b * a_stride
    const size_t a_stride = GATHER ? a_plane : (size_t)m_tiles * kPTileBytes;
    [[maybe_unused]] GatherOffsets<MT> gather;
    if constexpr (GATHER) {
        gather.load(a_rows + mt0 * 16, mt_count, wave, lane);
        // the zero bytes behind every tile of both buffers: no request writes them
        if (tid < 2 * MT * 4) *reinterpret_cast<uint32_t*>(a_lds + (tid >> 2) * kPTileBytes + kPZeroOff + (tid & 3) * 4) = 0u;
    }
    constexpr bool kByLane = MT > kMTilesMid && !PAIR && kWTilesPerWave == 1 && WT != kWtQ5;
    auto request_a = [&](int64_t b) {
        uint8_t* buf = a_lds + (b & 1) * kBufBytes;
        if constexpr (GATHER) request_a_rows<MT>(gather, a_src + (size_t)b * a_stride, buf, mt_count, wave, lane);
        else if constexpr (kByLane) request_a_tiles_by_lane<MT>(a_src + (size_t)b * a_stride, buf, copy_words, wave, lane);
        else request_a_tiles(a_src + (size_t)b * a_stride, buf, copy_words, wave, lane);
    };

    // Software pipeline over the super-blocks: while super-block b is multiplied, the activation tiles
    // of b+1 travel HBM/L2 -> LDS (other buffer) and this wave's weight tiles of b+1 travel into
    // registers.  One workgroup barrier per super-block.
    v4u seg0[kWTilesPerWave], seg1[kWTilesPerWave], hdr[kWTilesPerWave];
    v2u qh[kWTilesPerWave];
    v4u qh6[kWTilesPerWave];      // Q6_K: the top two bits of the codes; seg0 / seg1 hold its nibbles, hdr its sixteen scales
    uint32_t d6[kWTilesPerWave];  // Q6_K: fp16 d
    auto request_w = [&](int64_t b, int only = -1) {  // only >= 0: that tile alone
#pragma unroll
        for (int t = 0; t < kWTilesPerWave; ++t) {
            if (only >= 0 && t != only) continue;
            const uint8_t* tile = (PAIR && t == 1 ? w2 : w) + tile_offset(rt[t], b, nb, tile_stride<WT>());
            seg0[t] = load16(tile + lane * 16);
            seg1[t] = load16(tile + 1024 + lane * 16);
            if constexpr (Q6) {
                qh6[t] = load16(tile + kTile6HOff + lane * 16);
                hdr[t] = load16(tile + kTile6SOff + r * 16);
                d6[t] = *reinterpret_cast<const uint32_t*>(tile + kTile6DOff + r * 4);
            } else {
                hdr[t] = load16(tile + kTileQBytes + r * 16);
                if (Q5) qh[t] = *reinterpret_cast<const v2u*>(tile + kTileHBytes + lane * 8);
                else qh[t] = v2u{0u, 0u};
            }
        }
    };
    // K split over grid.z: this workgroup multiplies the super-blocks [b_begin, b_end) and writes its sums to
    // partial plane blockIdx.z (split_stride floats apart; the caller adds the planes in order)
    const int64_t b_begin = (int64_t)blockIdx.z * sb_split;
    const int64_t b_end = b_begin + sb_split < nb ? b_begin + sb_split : nb;
    y += (size_t)blockIdx.z * (size_t)split_stride;
    request_a(b_begin);
    request_w(b_begin);

    struct ATile {
        v4i a[4];
        v4f yd;
        v8h dg;
    };
    auto read_a = [&](ATile& t, const uint8_t* at) {
#pragma unroll
        for (int j = 0; j < 4; ++j) t.a[j] = *reinterpret_cast<const v4i*>(at + j * 1024 + lane * 16);
        t.yd = *reinterpret_cast<const v4f*>(at + kPScaleOff + kq * 16);
        if constexpr (!Q6) t.dg = *reinterpret_cast<const v8h*>(at + digit_off);
    };
    // The LDS operands of the next activation tile are requested while this one is multiplied.  One weight tile to a wavefront: by hand, the
    // 24 registers are there (kAhead).  Two: they are not (eight to twelve spill), but without a branch round every tile the compiler
    // finds room for them in turn (kAll: a workgroup whose tiles are all there; a form of its own for five, six, seven and eight).  Two
    // wavefronts to a SIMD waited 30 % of their time, much of it for these reads.  Against a read ahead of every tile's products, same
    // bits: 198 products of 64-row workgroups at 70 to 512 rows 0.951 of the time (Q4_K 2048 x 2048 at 128 rows 13.0 -> 12.1 us, Q5_K 4096 x 4096
    // at 100 rows 21.0 -> 19.0), 366 products and FFNs at 70 to 2048 rows 0.968 (Q4_K 14336 x 4096 at 700 rows 111 -> 99 us, Q6_K at
    // 2048 rows 0.96); least where the card's power is the limit (Q4_K from 1500 rows on: 0.98 to 1.0).  Without branches and without kAhead
    // one weight tile gains less and loses up to 9 % where the last column is short.  Q5_K's form of six tiles keeps the branches: without them
    // eight registers spill, and products with K in runs took up to 1.05 of the time with the branches of the form of eight (11088 x 6400 at 187
    // rows 61.0 -> 64.2 us); with its own it takes 0.987 of that time over 40 products and 0.961 over 24 pairs (61.4; pair 6832 x 1024 at 166 rows
    // 21.7 -> 20.3).
    constexpr bool kAhead = kDense && kWTilesPerWave == 1;
    constexpr int kFirst = MT != kMTilesMid || Q5 ? 0 : Q6 ? 2 : 1;
    auto multiply = [&](auto all_c) {
        constexpr bool kAll = decltype(all_c)::value;
        for (int64_t b = b_begin; b < b_end; ++b) {
            // everything this thread requested for super-block b has landed ...
            __builtin_amdgcn_s_waitcnt(0 | (0x7 << 4) | (0xF << 8));  // vmcnt(0)
            // ... and after the barrier so has everybody else's share of the activation tiles; every wave
            // is also done reading the other buffer (super-block b-1), which the next requests overwrite
            __syncthreads();
            if constexpr (PAIR && MT <= 4) {
                // Few activation tiles: the two weight tiles are expanded and multiplied one after the other, so that one
                // expanded tile is live at a time (38 registers less: three wavefronts per SIMD instead of two, which is
                // what a launch of many short workgroups needs); the activation operands are read from LDS once per tile.
                if (b + 1 < b_end) request_a(b + 1);
                const uint8_t* a_buf = a_lds + (b & 1) * kBufBytes;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    WTile w1;
                    if constexpr (Q6) expand_tile6(seg0[t], seg1[t], qh6[t], hdr[t], d6[t], kq, w1);
                    else expand_tile<Q5, kFifthChain<WT, MT>>(seg0[t], seg1[t], hdr[t], qh[t], kq, w1);
                    if (b + 1 < b_end) request_w(b + 1, t);  // the raw tile's registers are free again
                    // The first kFirst of a tile's four operands are read a tile ahead: as many as leave three wavefronts to a SIMD (none of Q5_K's).
                    // With the same in prefill_gemm_resident_kernel, 84 blocks of 31 to 158 rows per expert take 0.982 of the time (16 experts,
                    // top-4, 2816 x 768, Q6_K down at 180 tokens 60.5 -> 56.2 us; 256 + 1, top-8, 2048 x 512 at 1500 tokens: gate/up 116 -> 112, down 63.6 -> 63.4).
                    v4i first[2][kFirst + 1];
                    auto read_first = [&](v4i (&f)[kFirst + 1], const uint8_t* at) {
#pragma unroll
                        for (int j = 0; j < kFirst; ++j) f[j] = *reinterpret_cast<const v4i*>(at + j * 1024 + lane * 16);
                    };
                    read_first(first[0], a_buf);
#pragma unroll
                    for (int m = 0; m < MT; ++m) {
                        if (kAll || m < mt_count) {  // uniform over the workgroup
                            const uint8_t* at = a_buf + m * kPTileBytes;
                            ATile now;
#pragma unroll
                            for (int j = 0; j < 4; ++j) now.a[j] = j < kFirst ? first[m & 1][j < kFirst ? j : 0] : *reinterpret_cast<const v4i*>(at + j * 1024 + lane * 16);
                            if constexpr (!Q6) now.dg = *reinterpret_cast<const v8h*>(at + digit_off);
                            now.yd = *reinterpret_cast<const v4f*>(at + kPScaleOff + kq * 16);
                            if constexpr (kFirst > 0) {
                                if (m + 1 < MT) read_first(first[(m + 1) & 1], at + kPTileBytes);  // (past mt_count: read and not used)
                                __builtin_amdgcn_sched_barrier(0);  // ahead of this tile's products
                            }
                            const v4i (&a)[4] = now.a;
                            const float ydv[4] = {now.yd.x, now.yd.y, now.yd.z, now.yd.w};
                            const v4i zero = {0, 0, 0, 0};
                            const v4f zero_f = {0.0f, 0.0f, 0.0f, 0.0f};
                            v4i hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[0], w1.hi[0], zero, 0, 0, 0);
                            v4i lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[0], w1.lo[0], zero, 0, 0, 0);
                            v4i b5 = zero;
                            if constexpr (kFifthChain<WT, MT>) b5 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[0], w1.b5[0], zero, 0, 0, 0);
                            v4f mn = zero_f;
                            if constexpr (!Q6) mn = __builtin_amdgcn_mfma_f32_16x16x32_f16(now.dg, w1.mins, zero_f, 0, 0, 0);
#pragma unroll
                            for (int j = 1; j < 4; ++j) {
                                hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[j], w1.hi[j], hi, 0, 0, 0);
                                lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[j], w1.lo[j], lo, 0, 0, 0);
                                if constexpr (kFifthChain<WT, MT>) b5 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[j], w1.b5[j], b5, 0, 0, 0);
                            }
#pragma unroll
                            for (int i = 0; i < 4; ++i) {  // the arithmetic of the two-tiles-at-once form below
                                const int dot = join_digits<WT, MT>(hi[i], lo[i], b5[i]);
                                if constexpr (Q6) {
                                    acc[t][m][i] = __fmaf_rn(__fmul_rn(ydv[i], w1.d), (float)dot, acc[t][m][i]);
                                } else {
                                    const float v = __fmaf_rn(-w1.dmin, mn[i], __fmul_rn(w1.d, (float)dot));
                                    acc[t][m][i] = __fmaf_rn(ydv[i], v, acc[t][m][i]);
                                }
                            }
                        }
                    }
                }
                continue;
            }
            WTile wt[kWTilesPerWave];
#pragma unroll
            for (int t = 0; t < kWTilesPerWave; ++t) {
                if constexpr (Q6) expand_tile6(seg0[t], seg1[t], qh6[t], hdr[t], d6[t], kq, wt[t]);
                else expand_tile<Q5, kFifthChain<WT, MT>>(seg0[t], seg1[t], hdr[t], qh[t], kq, wt[t]);
            }
            if (b + 1 < b_end) {
                request_a(b + 1);
                request_w(b + 1);
            }
            const uint8_t* a_buf = a_lds + (b & 1) * kBufBytes;

            ATile at[kAhead ? 2 : 1];
            if constexpr (kAhead) read_a(at[0], a_buf);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (kAll || m < mt_count) {  // uniform over the workgroup
                    if constexpr (kAhead) {
                        if (m + 1 < MT) read_a(at[(m + 1) & 1], a_buf + (m + 1) * kPTileBytes);  // (past mt_count: read and not used)
                        __builtin_amdgcn_sched_barrier(0);  // ahead of this tile's products
                    } else {
                        read_a(at[0], a_buf + m * kPTileBytes);
                    }
                    const ATile& now = at[kAhead ? m & 1 : 0];
                    const v4i (&a)[4] = now.a;
                    const float ydv[4] = {now.yd.x, now.yd.y, now.yd.z, now.yd.w};
                    const v8h dg = now.dg;
                    const v4i zero = {0, 0, 0, 0};
                    const v4f zero_f = {0.0f, 0.0f, 0.0f, 0.0f};
                    v4i hi[kWTilesPerWave], lo[kWTilesPerWave], b5[kWTilesPerWave];
                    v4f mn[kWTilesPerWave];
#pragma unroll
                    for (int t = 0; t < kWTilesPerWave; ++t) {
                        hi[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[0], wt[t].hi[0], zero, 0, 0, 0);
                        lo[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[0], wt[t].lo[0], zero, 0, 0, 0);
                        b5[t] = zero;
                        if constexpr (kFifthChain<WT, MT>) b5[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[0], wt[t].b5[0], zero, 0, 0, 0);
                        if constexpr (!Q6) mn[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(dg, wt[t].mins, zero_f, 0, 0, 0);
                    }
#pragma unroll
                    for (int j = 1; j < 4; ++j)
#pragma unroll
                        for (int t = 0; t < kWTilesPerWave; ++t) {
                            hi[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[j], wt[t].hi[j], hi[t], 0, 0, 0);
                            lo[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[j], wt[t].lo[j], lo[t], 0, 0, 0);
                            if constexpr (kFifthChain<WT, MT>) b5[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[j], wt[t].b5[j], b5[t], 0, 0, 0);
                        }
#pragma unroll
                    for (int t = 0; t < kWTilesPerWave; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int dot = join_digits<WT, MT>(hi[t][i], lo[t][i], b5[t][i]);
                            if constexpr (Q6) {
                                // the integer of the reference's kernel (times 4, taken out of d), then its one fused multiply-add
                                // per block (core/src/llm/matmul/q6_small_batch.h:84-86)
                                acc[t][m][i] = __fmaf_rn(__fmul_rn(ydv[i], wt[t].d), (float)dot, acc[t][m][i]);
                            } else {
                                // yd * (d * dot - dmin * min_dot): three fp32 operations per output and super-block
                                const float v = __fmaf_rn(-wt[t].dmin, mn[t][i], __fmul_rn(wt[t].d, (float)dot));
                                acc[t][m][i] = __fmaf_rn(ydv[i], v, acc[t][m][i]);
                            }
                        }
                }
            }
        }
    };
    if constexpr (kDense && kWTilesPerWave == 2 && !(Q5 && MT == 6)) {
        if (mt_count == MT) multiply(std::true_type{});
        else multiply(std::false_type{});
    } else {
        multiply(std::false_type{});
    }

    if constexpr (PAIR) {  // one output per (token, row): silu(gate) * up
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[0][m][i] = silu_mul(acc[0][m][i], acc[1][m][i], silu_mode);
    }
    constexpr int kStoredTiles = PAIR ? 1 : kWTilesPerWave;
    if (out_rows) {  // grouped down product: row 16 (mt0 + m) + 4 kq + i of the plan goes to row out_rows[..] of y (-1: padding)
#pragma unroll
        for (int t = 0; t < kStoredTiles; ++t) {
            const int64_t row = (rt0 + t) * kTileRows + r;
            if (rt0 + t >= rowtiles || row >= rows) continue;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (m >= mt_count) continue;
                const int4 dst = *reinterpret_cast<const int4*>(out_rows + (mt0 + m) * 16 + kq * 4);
                const int dsts[4] = {dst.x, dst.y, dst.z, dst.w};
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (dsts[i] >= 0) y[(size_t)dsts[i] * (size_t)ldy + row] = acc[t][m][i];
            }
        }
        return;
    }
    // Stores: lane (r, kq) holds weight row r of its tiles for the tokens 16 m + 4 kq + i.  One pointer per lane walks
    // down the token rows (an addition per store, no product).
    const int tok_left = (int)(n_tokens - mt0 * 16) - kq * 4;  // tokens from this lane's first one to the end
#pragma unroll
    for (int t = 0; t < kStoredTiles; ++t) {
        const int64_t row = (rt0 + t) * kTileRows + r;
        if (rt0 + t >= rowtiles || row >= rows) continue;
        float* yp = y + (mt0 * 16 + kq * 4) * ldy + row;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (m < mt_count && m * 16 + i < tok_left) *yp = acc[t][m][i];
                yp += ldy;
            }
            yp += 12 * ldy;
        }
    }
}

// The expert-grouped product over rows of a few super-blocks (the down experts of a MoE block: two super-blocks of 512 columns):
// a workgroup stages ALL super-blocks of its item's activation tiles once and walks row_blocks blocks of 64 weight rows with them --
// one barrier, and the first tiles of a block travel while the block before it is multiplied.  Same arithmetic as above.
template <int WT, int MT>
__global__ void __launch_bounds__(256, 3) prefill_gemm_resident_kernel(const uint8_t* __restrict__ w, int rowtiles, int64_t rows, int nb,
                                                                       const uint8_t* __restrict__ ap, int64_t m_tiles, float* __restrict__ y, int64_t ldy,
                                                                       const int32_t* __restrict__ plan, int64_t expert_bytes,
                                                                       const int32_t* __restrict__ out_rows, const uint8_t* __restrict__ w_shared, int row_blocks) {
    extern __shared__ __align__(16) uint8_t a_lds[];  // nb buffers of MT * kPTileBytes bytes, then the output row of each of the tiles' rows
    constexpr int kBufBytes = MT * kPTileBytes;
    constexpr bool Q5 = WT == kWtQ5, Q6 = WT == kWtQ6;
    constexpr int kFirst = MT == kMTilesMid && !Q5 ? 2 : 0;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kq = lane >> 4;
    const int item = blockIdx.y;
    if (item >= plan[0]) return;  // the whole workgroup, before any barrier
    const int expert = plan[4 + 3 * item];  // -1: the shared expert's rows
    const int64_t mt0 = plan[5 + 3 * item];
    const int mt_count = plan[6 + 3 * item];
    w = expert < 0 ? w_shared : w + (size_t)expert * (size_t)expert_bytes;
    int rt = (int)blockIdx.x * 4 * row_blocks + wave;
    const int rt_end = ((int)blockIdx.x + 1) * 4 * row_blocks < rowtiles ? ((int)blockIdx.x + 1) * 4 * row_blocks : rowtiles;
    v4u seg0, seg1, hdr, qh6;
    v2u qh = {0u, 0u};
    uint32_t d6 = 0;
    auto request_w = [&](int t, int b) {
        const uint8_t* tile = w + tile_offset(t, b, nb, tile_stride<WT>());
        seg0 = load16(tile + lane * 16);
        seg1 = load16(tile + 1024 + lane * 16);
        if constexpr (Q6) {
            qh6 = load16(tile + kTile6HOff + lane * 16);
            hdr = load16(tile + kTile6SOff + r * 16);
            d6 = *reinterpret_cast<const uint32_t*>(tile + kTile6DOff + r * 4);
        } else {
            hdr = load16(tile + kTileQBytes + r * 16);
            if constexpr (Q5) qh = *reinterpret_cast<const v2u*>(tile + kTileHBytes + lane * 8);
        }
    };
    for (int b = 0; b < nb; ++b)
        request_a_tiles(ap + ((size_t)b * (size_t)m_tiles + (size_t)mt0) * kPTileBytes, a_lds + b * kBufBytes, mt_count * kPTileWords, wave, lane);
    if (rt < rt_end) request_w(rt, 0);
    int32_t* dst_lds = reinterpret_cast<int32_t*>(a_lds + nb * kBufBytes);
    if (tid < mt_count * 16) dst_lds[tid] = out_rows ? out_rows[mt0 * 16 + tid] : (int)mt0 * 16 + tid;  // -1: padding
    __builtin_amdgcn_s_waitcnt(0 | (0x7 << 4) | (0xF << 8));  // vmcnt(0): this thread's share of the tiles has landed ...
    __syncthreads();                                          // ... and everybody else's; nothing below writes LDS
    const int digit_off = kq < 2 ? kPDigitOff + r * 32 + kq * 16 : kPZeroOff;
    for (; rt < rt_end; rt += 4) {
        float acc[MT][4];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[m][i] = 0.0f;
        for (int b = 0; b < nb; ++b) {
            WTile wt;
            if constexpr (Q6) expand_tile6(seg0, seg1, qh6, hdr, d6, kq, wt);
            else expand_tile<Q5, kFifthChain<WT, MT>>(seg0, seg1, hdr, qh, kq, wt);
            // (ahead of this block's stores: waiting for a tile then never waits for them)
            if (b + 1 < nb) request_w(rt, b + 1);
            else if (rt + 4 < rt_end) request_w(rt + 4, 0);
            const uint8_t* a_buf = a_lds + b * kBufBytes;
            v4i first[2][kFirst + 1];  // the first kFirst of a tile's four operands, one tile ahead
            auto read_first = [&](v4i (&f)[kFirst + 1], const uint8_t* at) {
#pragma unroll
                for (int j = 0; j < kFirst; ++j) f[j] = *reinterpret_cast<const v4i*>(at + j * 1024 + lane * 16);
            };
            read_first(first[0], a_buf);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (m < mt_count) {  // uniform over the workgroup
                    const uint8_t* at = a_buf + m * kPTileBytes;
                    v4i a[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) a[j] = j < kFirst ? first[m & 1][j < kFirst ? j : 0] : *reinterpret_cast<const v4i*>(at + j * 1024 + lane * 16);
                    const float4 yd = *reinterpret_cast<const float4*>(at + kPScaleOff + kq * 16);
                    v8h dg;
                    if constexpr (!Q6) dg = *reinterpret_cast<const v8h*>(at + digit_off);
                    if constexpr (kFirst > 0) {
                        if (m + 1 < MT) read_first(first[(m + 1) & 1], at + kPTileBytes);  // (past mt_count: read and not used)
                        __builtin_amdgcn_sched_barrier(0);  // ahead of this tile's products
                    }
                    const float ydv[4] = {yd.x, yd.y, yd.z, yd.w};
                    const v4i zero = {0, 0, 0, 0};
                    const v4f zero_f = {0.0f, 0.0f, 0.0f, 0.0f};
                    v4i hi = zero, lo = zero, b5 = zero;
                    v4f mn = zero_f;
                    if constexpr (!Q6) mn = __builtin_amdgcn_mfma_f32_16x16x32_f16(dg, wt.mins, zero_f, 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[j], wt.hi[j], hi, 0, 0, 0);
                        lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[j], wt.lo[j], lo, 0, 0, 0);
                        if constexpr (kFifthChain<WT, MT>) b5 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[j], wt.b5[j], b5, 0, 0, 0);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int dot = join_digits<WT, MT>(hi[i], lo[i], b5[i]);
                        if constexpr (Q6) {
                            acc[m][i] = __fmaf_rn(__fmul_rn(ydv[i], wt.d), (float)dot, acc[m][i]);
                        } else {
                            const float v = __fmaf_rn(-wt.dmin, mn[i], __fmul_rn(wt.d, (float)dot));
                            acc[m][i] = __fmaf_rn(ydv[i], v, acc[m][i]);
                        }
                    }
                }
            }
        }
        const int64_t row = (int64_t)rt * kTileRows + r;
        if (row < rows) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (m >= mt_count) continue;
                const int4 dst = *reinterpret_cast<const int4*>(dst_lds + m * 16 + kq * 4);
                const int dsts[4] = {dst.x, dst.y, dst.z, dst.w};
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (dsts[i] >= 0) y[(size_t)dsts[i] * (size_t)ldy + row] = acc[m][i];
            }
        }
    }
}

// One workgroup per (tile of 16 activation rows, super-block): its four wavefronts quantize four rows each into an
// image of the tile in LDS, which then leaves as one run of 16-byte stores (a wavefront per row writing straight to
// the tile scattered its 256 bytes over 32 cache lines: 52 us for the 16384 gathered rows of a MoE block at 2048
// tokens).  Rows in [n, 16 * m_tiles) are written as zeros.
// kSwiglu: the row is silu(x) * x2 of two inputs (the gate and up products of an FFN), formed here instead of in a
// pass of its own; h_out, if given, receives it as fp32 as well.
// Expert-grouped forms: plan (tiles past plan[1] are skipped), row_src (row m of the tiles is row row_src[m] of x, -1:
// padding, zeros), h_rows (row m of the tiles is row h_rows[m] of h_out, -1: not written).
// kRowsPerWave: four (256 threads) in general; one (1024 threads, a wavefront per row) for launches of a few workgroups
// (sixteen rows: one workgroup per super-block), where the four rows one after the other are the launch's length.
template <bool kSwiglu, int kRowsPerWave = 4>
__global__ void __launch_bounds__(64 * 16 / kRowsPerWave) quantize_q8k_pmajor_kernel(const float* __restrict__ x, const float* __restrict__ x2,
                                                                  int silu_mode, float* __restrict__ h_out, int64_t ldh,
                                                                  int64_t n, int64_t ldx, int64_t nb, int64_t m_tiles,
                                                                  uint8_t* __restrict__ ap, const int32_t* __restrict__ plan,
                                                                  const int32_t* __restrict__ row_src,
                                                                  const int32_t* __restrict__ h_rows) {
    __shared__ __align__(16) uint8_t img[kPTileBytes];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t tile = blockIdx.x, b = blockIdx.y;
    if (plan && tile >= (int64_t)plan[1]) return;  // the whole workgroup, before the barrier
    if (plan && kSwiglu && tile >= (int64_t)plan[2]) silu_mode = plan[3];  // the shared expert's tiles: its own SiLU form
    constexpr int kThreads = 64 * 16 / kRowsPerWave;
    int64_t src[kRowsPerWave], hr[kRowsPerWave];
    float4 v[kRowsPerWave], u[kRowsPerWave];
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
        const int64_t m = tile * 16 + wave * kRowsPerWave + r;
        src[r] = row_src ? row_src[m] : (m < n ? m : -1);
        hr[r] = h_rows ? h_rows[m] : src[r];
    }
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {  // all of the wavefront's rows are requested before any is worked on
        const int64_t from = src[r] >= 0 ? src[r] : 0;
        v[r] = *reinterpret_cast<const float4*>(x + from * ldx + b * kQK + lane * 4);
        if (kSwiglu) u[r] = *reinterpret_cast<const float4*>(x2 + from * ldx + b * kQK + lane * 4);
    }
    // elements 4*lane..4*lane+3: sub-block g = lane/8, elements 4*(lane%8).. of it
    const int g = lane >> 3;
    const int j = 2 * (g >> 2) + (g & 1), half = (g >> 1) & 1;
    const int kq = (lane & 7) >> 1;
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
        const int tok = wave * kRowsPerWave + r;
        float e[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (src[r] >= 0) {  // wave-uniform
            e[0] = v[r].x, e[1] = v[r].y, e[2] = v[r].z, e[3] = v[r].w;
            if (kSwiglu) {
                e[0] = silu_mul(e[0], u[r].x, silu_mode), e[1] = silu_mul(e[1], u[r].y, silu_mode);
                e[2] = silu_mul(e[2], u[r].z, silu_mode), e[3] = silu_mul(e[3], u[r].w, silu_mode);
                if (h_out && hr[r] >= 0)
                    *reinterpret_cast<float4*>(h_out + hr[r] * ldh + b * kQK + lane * 4) = float4{e[0], e[1], e[2], e[3]};
            }
        }
        const Q8Lane q = quantize_block_q8k(e, lane);
        *reinterpret_cast<uint32_t*>(img + j * 1024 + (kq * 16 + tok) * 16 + half * 8 + (lane & 1) * 4) = q.packed;
        const int bs = q.bsum + __shfl_xor(q.bsum, 4, 64);  // codes 32g .. 32g+31
        if ((lane & 7) == 0) {  // bs = 128 h + l, both parts exact in fp16
            _Float16* digits = reinterpret_cast<_Float16*>(img + kPDigitOff + tok * 32);
            digits[g] = (_Float16)(float)(bs & 127);
            digits[8 + g] = (_Float16)(float)((bs >> 7) * 128);
        }
        if (lane == 0) *reinterpret_cast<float*>(img + kPScaleOff + tok * 4) = q.d;
    }
    if (tid < 4) *reinterpret_cast<uint32_t*>(img + kPZeroOff + tid * 4) = 0u;
    __syncthreads();
    v4u* dst = reinterpret_cast<v4u*>(ap + ((size_t)b * (size_t)m_tiles + (size_t)tile) * kPTileBytes);
    for (int i = tid; i < kPTileWords; i += kThreads) dst[i] = reinterpret_cast<const v4u*>(img)[i];
}

// Rows that are gathered to several places (a token is a row of top_k experts, and of the shared one) are quantized once, into the
// row layout (pmajor.h), from where the expert-grouped GEMM fetches them.  A wavefront per (row, super-block).
__device__ __forceinline__ void quantize_prow(const GroupedRows& rows, int64_t row, int64_t b, int lane) {
    const float4 v = *reinterpret_cast<const float4*>(rows.x + row * rows.ldx + b * kQK + lane * 4);
    const float e[4] = {v.x, v.y, v.z, v.w};
    const Q8Lane q = quantize_block_q8k(e, lane);
    uint8_t* dst = rows.out + ((size_t)b * (size_t)rows.n + (size_t)row) * kPRowBytes;
    // elements 4*lane..4*lane+3: sub-block g = lane/8, elements 4*(lane%8).. of it
    const int g = lane >> 3, j = 2 * (g >> 2) + (g & 1), half = (g >> 1) & 1, kq = (lane & 7) >> 1;
    *reinterpret_cast<uint32_t*>(dst + j * 64 + kq * 16 + half * 8 + (lane & 1) * 4) = q.packed;
    const int bs = q.bsum + __shfl_xor(q.bsum, 4, 64);  // codes 32g .. 32g+31
    if ((lane & 7) == 0) {  // bs = 128 h + l, both parts exact in fp16
        _Float16* digits = reinterpret_cast<_Float16*>(dst + kPRowDigitOff);
        digits[g] = (_Float16)(float)(bs & 127);
        digits[8 + g] = (_Float16)(float)((bs >> 7) * 128);
    }
    if (lane == 0) *reinterpret_cast<float*>(dst + kPRowScaleOff) = q.d;
}

// A workgroup of 1024 threads, number wg of wgs: sixteen rows of a super-block, one per wavefront, and again as many workgroups further
__device__ __forceinline__ void quantize_prow_runs(const GroupedRows& rows, uint32_t wg, uint32_t wgs) {
    const uint32_t per_block = (uint32_t)((rows.n + 15) / 16), runs = per_block * (uint32_t)rows.nb;  // < 2^31: host-checked
    for (uint32_t q = wg; q < runs; q += wgs) {
        const uint32_t b = q / per_block;
        const int64_t row = (int64_t)(q - b * per_block) * 16 + (threadIdx.x >> 6);
        if (row < rows.n) quantize_prow(rows, row, b, threadIdx.x & 63);
    }
}

// y[tok][row] = plane 0 + plane 1 + ... in that order; four rows per thread, the planes' rows `pitch` floats apart (rows padded to four:
// what lies in the padding is read and not stored)
__global__ void __launch_bounds__(256) prefill_sum_planes_kernel(const float* __restrict__ part, int splits, int64_t n, int64_t rows, int64_t pitch,
                                                                 float* __restrict__ y, int64_t ldy) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (token, group of four rows)
    const int64_t per_row = pitch >> 2;
    if (i >= n * per_row) return;
    const int64_t tok = i / per_row, q = i - tok * per_row;
    const float4* src = reinterpret_cast<const float4*>(part + (size_t)tok * pitch) + q;
    float4 acc = src[0];
    for (int z = 1; z < splits; ++z) {
        const float4 v = src[(size_t)z * (size_t)(n * per_row)];
        acc.x = __fadd_rn(acc.x, v.x), acc.y = __fadd_rn(acc.y, v.y), acc.z = __fadd_rn(acc.z, v.z), acc.w = __fadd_rn(acc.w, v.w);
    }
    float* dst = y + tok * ldy + q * 4;
    const int64_t left = rows - q * 4;
    dst[0] = acc.x;
    if (left > 1) dst[1] = acc.y;
    if (left > 2) dst[2] = acc.z;
    if (left > 3) dst[3] = acc.w;
}

// Shape of a launch: 128- or 64-row workgroups, the activation tiles in `groups` workgroup columns of tiles_per_wg <= 8, K in
// `splits` runs of super-blocks (planes of partial sums that a second launch adds in order).  A compute unit holds two workgroups,
// and a workgroup walks its super-blocks one after the other, so what counts is how long a workgroup takes and how the workgroups
// fill the 2 x compute_units() slots.  Pace: us a workgroup takes for t activation tiles and sb super-blocks,
//     two on a unit  sb (sb2 + tile2 t) + fix2 + store t        one alone  sb (sb1 + tile1 t) + fix1 + store t
// (fix, store: first tiles, last stores); load: what every unit being busy costs on top, per tile of a round of slots; the workgroups
// that a full round leaves take later1 / later2 of that (up to one per unit / more: the rounds do not end at one time); a
// workgroup beside one of x of its length is held up by x^3 of the difference (half as long: an eighth, since the short ones pile up
// on units of their own first).  Least-squares fits over every shape of 8,650 dense products and 3,270 gate/up pairs (512 to 16,384
// rows, 4 to 56 super-blocks, 48 to 2048 tokens; residuals 4 and 2.5 %), 128 rows | 64 rows | pair:
struct Pace {
    float sb2, tile2, sb1, tile1, fix2, store, fix1, load, later1, later2;
};
enum { kWide, kNarrow, kPairForm };
constexpr Pace kPace[3][3] = {
    {{0.870f, 0.267f, 0.505f, 0.213f, 1.07f, 0.020f, 0.81f, 0.112f, 0.815f, 0.973f},   // Q4_K
     {0.511f, 0.143f, 0.353f, 0.143f, 0.38f, 0.000f, 0.00f, 0.075f, 0.917f, 1.011f},
     {0.901f, 0.332f, 0.579f, 0.242f, 3.85f, 0.000f, 2.50f, 0.044f, 0.893f, 1.030f}},
    {{1.565f, 0.263f, 0.898f, 0.198f, 1.20f, 0.024f, 0.92f, 0.138f, 0.768f, 0.941f},   // Q5_K: 16-bit products cost the expansion
     {0.823f, 0.148f, 0.487f, 0.153f, 0.34f, 0.002f, 0.00f, 0.080f, 0.893f, 1.004f},
     {1.721f, 0.323f, 1.050f, 0.233f, 2.85f, 0.000f, 0.93f, 0.037f, 0.891f, 1.015f}},
    {{1.626f, 0.230f, 0.956f, 0.177f, 1.19f, 0.021f, 0.70f, 0.129f, 0.763f, 0.938f},   // Q6_K: no min MFMA
     {0.897f, 0.121f, 0.480f, 0.122f, 0.28f, 0.000f, 0.00f, 0.071f, 0.868f, 0.988f},
     {1.759f, 0.285f, 1.061f, 0.211f, 3.10f, 0.000f, 0.95f, 0.051f, 0.916f, 1.029f}}};

GemmShape shape_of(int form, int64_t rows, int64_t nb, int64_t m_tiles, int64_t t, int64_t splits) {
    const int64_t rowtiles = (rows + 15) / 16;
    GemmShape s;
    s.narrow = form == kNarrow, s.tiles_per_wg = (int)t;
    s.row_wgs = (unsigned)(form == kWide ? (rowtiles + 7) / 8 : (rowtiles + 3) / 4), s.groups = (unsigned)((m_tiles + t - 1) / t);
    s.sb_split = (int)((nb + splits - 1) / splits);
    s.splits = (int)((nb + s.sb_split - 1) / s.sb_split);  // every run holds a super-block
    return s;
}

// us of a launch, its planes included
float shape_us(const Pace& p, const GemmShape& s, int64_t rows, int64_t nb, int64_t m_tiles, int64_t n) {
    const int64_t units = compute_units(), slots = 2 * units;
    const double per_slot = 1.0 / (double)slots;
    auto rounds = [&](int64_t x) { return (int64_t)(((double)x + 0.5) * per_slot); };  // x / slots without a division
    const int64_t t = s.tiles_per_wg, sb = s.sb_split, wgs = (int64_t)s.row_wgs * s.groups * s.splits;
    auto two = [&](int64_t b, int64_t k) { return (float)b * (p.sb2 + p.tile2 * (float)k) + p.fix2 + p.store * (float)k; };
    auto one = [&](int64_t b, int64_t k) {
        const float v = (float)b * (p.sb1 + p.tile1 * (float)k) + p.fix1 + p.store * (float)k, w = two(b, k);
        return v < w ? v : w;
    };
    auto rest = [&](int64_t r, bool later, int64_t b, int64_t k) {  // r < slots workgroups that a full round leaves, or the only ones
        if (r == 0) return 0.0f;
        return r <= units ? (later ? p.later1 : 1.0f) * one(b, k) : (later ? p.later2 : 1.0f) * two(b, k);
    };
    // dispatched last, and shorter: the last run of an uneven K split, else the last column
    const int64_t b_last = s.splits > 1 ? nb - (s.splits - 1) * sb : sb, t_last = s.splits > 1 ? t : m_tiles - (int64_t)(s.groups - 1) * t;
    const int64_t shorter = wgs > (int64_t)s.row_wgs && (b_last < sb || t_last < t) ? (int64_t)s.row_wgs * (s.splits > 1 ? s.groups : 1) : 0;
    const int64_t full = rounds(wgs - shorter), r = wgs - shorter - full * slots, spare = slots - r;
    const float l2 = two(sb, t);
    float us = (float)full * l2;
    if (shorter == 0) {
        us += rest(r, full > 0, sb, t);
    } else if (r == 0) {
        const int64_t more = rounds(shorter);
        us += (float)more * two(b_last, t_last) + rest(shorter - more * slots, true, b_last, t_last);
    } else {
        const float s2 = two(b_last, t_last);
        if (shorter <= spare) {
            const float l1 = one(sb, t), s1 = one(b_last, t_last);
            const float x = s2 < l2 ? s2 / l2 : 1.0f;
            float tail = r > units ? l2 : r + shorter > units ? l1 + (l2 - l1) * x * x * x : l1;
            if (full > 0) tail *= r > units ? p.later2 : p.later1;
            us += tail > s1 ? tail : s1;
        } else {
            const float chain = (float)((shorter + spare - 1) / spare) * s2;
            int64_t beside = (int64_t)(l2 / s2);
            beside = (beside < 1 ? 1 : beside) * spare;
            const int64_t left = shorter > beside ? shorter - beside : 0;
            const int64_t more = rounds(left);
            const float after = l2 + (float)more * s2 + rest(left - more * slots, true, b_last, t_last);
            const float tail = chain < after ? chain : after;
            us += tail > l2 ? tail : l2;
        }
    }
    us += p.load * (float)(sb * s.splits) * (float)((int64_t)s.row_wgs * m_tiles) / (float)slots;
    if (s.splits > 1) us += 2.8f + 0.55e-6f * (float)s.splits * (float)(n * rows);  // a launch, the planes written and read
    return us;
}

// The plain shape -- 64-row workgroups up to one 128-row workgroup per unit, tiles in eights, K in as many runs as fill the slots --
// unless the estimate of another one is less by kLess.  Over the fitted products Q4_K / Q5_K / Q6_K the chosen shape takes 1.007 /
// 1.010 / 1.009 of the fastest one's time (pairs 1.003 / 1.002 / 1.003), the plain shape 1.115 / 1.094 / 1.080 (pairs 1.16 / 1.12 /
// 1.11); the choice is over 5 % slower than plain on 0.2 / 0.5 / 1.2 % of the products, 0.4 / 1.0 / 1.4 % at a kLess of 0.98.
// 4096 x 14336 at 130 / 391 / 700 / 1200 rows against the plain shape, with quantizer and planes: 46 / 84 / 145 / 245 ->
// 37 / 70 / 119 / 203 us, 14336 x 4096 at 130 / 391 / 700 39 / 74 / 116 -> 31 / 67 / 109.
constexpr float kLess = 0.97f, kLessPair = 0.95f;
GemmShape choose_shape(const Pace* pace, bool pair, int64_t rows, int64_t nb, int64_t n) {
    const int64_t units = compute_units(), m_tiles = (n + 15) / 16, rowtiles = (rows + 15) / 16;
    const int64_t most = m_tiles < kMTilesPerGroup ? m_tiles : kMTilesPerGroup, min_groups = (m_tiles + kMTilesPerGroup - 1) / kMTilesPerGroup;
    const int64_t max_splits = pair || (rows & 3) ? 1 : (nb / 4 < 1 ? 1 : nb / 4 < 16 ? nb / 4 : 16);  // at least four super-blocks per run
    const int plain_form = pair ? kPairForm : (rowtiles + 7) / 8 * min_groups <= units ? kNarrow : kWide;
    GemmShape plain = shape_of(plain_form, rows, nb, m_tiles, most, 1);
    const int64_t fill = 2 * units / ((int64_t)plain.row_wgs * plain.groups), runs = fill < nb / 4 ? fill : nb / 4;
    if (!pair && !(rows & 3) && runs > 1) plain = shape_of(plain_form, rows, nb, m_tiles, most, runs);
    plain.us = shape_us(pace[plain_form], plain, rows, nb, m_tiles, n);
    GemmShape best = plain;
    for (int form = pair ? kPairForm : kWide; form <= (pair ? kPairForm : kNarrow); ++form) {
        const Pace& p = pace[form];
        int64_t before = 0;
        for (int64_t want = min_groups; want < min_groups + 6; ++want) {
            const int64_t t = want < min_groups + 5 ? (m_tiles + want - 1) / want : most;  // dealt evenly; in eights with a short column
            if (t == before) continue;
            before = t;
            GemmShape s = shape_of(form, rows, nb, m_tiles, t, 1);
            for (int sp = 1; sp <= max_splits; ++sp) {
                s.sb_split = ((int)nb + sp - 1) / sp, s.splits = ((int)nb + s.sb_split - 1) / s.sb_split;
                // (no longer than the best so far even as workgroups alone; a count that leaves no empty run)
                if ((float)s.sb_split * (p.sb1 + p.tile1 * (float)t) < best.us && s.splits == sp) {
                    s.us = shape_us(p, s, rows, nb, m_tiles, n);
                    if (s.us < best.us) best = s;
                }
                if ((int64_t)s.row_wgs * s.groups * sp > 4 * units) break;  // two rounds and more: further runs only add planes
            }
        }
    }
    return best.us <= (pair ? kLessPair : kLess) * plain.us ? best : plain;
}

// ---- expert-grouped GEMM: the plan ------------------------------------------------------------------------
// Every workgroup repeats the (short) prefix sums over the groups and then takes its share of the items and rows:
// each row costs two dependent reads of the entry lists, so one workgroup alone needs 29 us for 2048 tokens.
// From the expert groups of the routing (entries sorted by expert: group g holds the entries
// group_begin[g] .. group_begin[g + 1] - 1 of expert group_expert[g]) it lays the entries out in tiles of 16 rows, every
// group starting a new tile, and cuts every group's tiles into items of up to eight tiles, the unit a GEMM workgroup
// column multiplies.  plan: [0] items, [1] tiles, [4 + 3 i ..] = (expert, first tile, tiles) of item i; row_src[r] /
// out_row[r] for row r of the tiles: the token whose activations it holds and the row of the per-(token, slot) output
// it produces (token * slots + k), -1 for padding (src_per_slot: the activations are per (token, slot) rows too).
// Workgroups past plan_wgs quantize the rows that the GEMM will gather: the plan is a chain of short dependent steps on a few compute
// units, and the rows need nothing of it (256 + 1 experts, 2048 columns, 1500 tokens: 5.4 + 5.7 us as two launches, 6.9 as one;
// the block 235.9 -> 230.9).
__global__ void __launch_bounds__(1024) moe_gemm_plan_kernel(const int32_t* __restrict__ n_groups, const int32_t* __restrict__ group_expert,
                                                             const int32_t* __restrict__ group_begin,
                                                             const int32_t* __restrict__ entry_token,
                                                             const int32_t* __restrict__ entry_k, int slots, int src_per_slot,
                                                             int groups_max, int sh_tokens, int sh_slot, int sh_silu_mode,
                                                             int32_t* __restrict__ plan, int32_t* __restrict__ row_src,
                                                             int32_t* __restrict__ out_row, int mt, int plan_wgs, GroupedRows rows) {
    if ((int)blockIdx.x >= plan_wgs) {
        quantize_prow_runs(rows, blockIdx.x - (uint32_t)plan_wgs, gridDim.x - (uint32_t)plan_wgs);
        return;
    }
    extern __shared__ int32_t plan_sh[];  // begin[g], tile0[g], item0[g]: groups_max + 2 each
    int32_t* begin = plan_sh;
    int32_t* tile0 = begin + groups_max + 2;
    int32_t* item0 = tile0 + groups_max + 2;
    const int tid = threadIdx.x, nt = blockDim.x;
    // sh_tokens > 0: one more group behind the routed ones, the shared expert with every token in order (expert -1,
    // output slot sh_slot); plan[2] = its first tile, plan[3] = its SiLU form
    const int ng_routed = *n_groups < groups_max ? *n_groups : groups_max;
    const int ng = ng_routed + (sh_tokens > 0 ? 1 : 0);
    for (int g = tid; g <= ng_routed; g += nt) begin[g] = group_begin[g];
    __syncthreads();
    if (tid == 0 && sh_tokens > 0) begin[ng] = begin[ng_routed] + sh_tokens;
    __syncthreads();
    if (tid < 64) {  // wavefront 0: exclusive prefix sums of tiles and items, lane l over a run of consecutive groups
        const int per = (ng + 63) / 64, g0 = tid * per;
        int tiles = 0, items = 0;
        for (int g = g0; g < g0 + per && g < ng; ++g) {
            const int t = (begin[g + 1] - begin[g] + 15) >> 4;
            tiles += t, items += (t + mt - 1) / mt;
        }
        int ts = tiles, is = items;  // inclusive scans across the lanes
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int a = __shfl_up(ts, d, 64), b = __shfl_up(is, d, 64);
            if (tid >= d) ts += a, is += b;
        }
        const int all_tiles = __shfl(ts, 63, 64), all_items = __shfl(is, 63, 64);
        ts -= tiles, is -= items;
        for (int g = g0; g < g0 + per && g < ng; ++g) {
            const int t = (begin[g + 1] - begin[g] + 15) >> 4;
            tile0[g] = ts, item0[g] = is;
            ts += t, is += (t + mt - 1) / mt;
        }
        if (tid == 0) {
            tile0[ng] = all_tiles, item0[ng] = all_items;
        }
    }
    __syncthreads();
    if (tid == 0 && blockIdx.x == 0)
        plan[0] = item0[ng], plan[1] = tile0[ng], plan[2] = sh_tokens > 0 ? tile0[ng_routed] : tile0[ng], plan[3] = sh_silu_mode;
    // the group of position q in a non-decreasing prefix array: the last g with first[g] <= q (empty groups cannot occur)
    auto group_of = [&](const int32_t* first, int q) {
        int lo = 0, hi = ng - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (first[mid] <= q) lo = mid;
            else hi = mid - 1;
        }
        return lo;
    };
    const int tiles = tile0[ng], items = item0[ng];
    const int first = blockIdx.x * nt + tid, step = plan_wgs * nt;
    for (int i = first; i < items; i += step) {
        const int g = group_of(item0, i);
        const int t_g = tile0[g + 1] - tile0[g], at = (i - item0[g]) * mt;
        plan[4 + 3 * i] = g < ng_routed ? group_expert[g] : -1;
        plan[5 + 3 * i] = tile0[g] + at;
        plan[6 + 3 * i] = t_g - at < mt ? t_g - at : mt;
    }
    for (int rr = first; rr < tiles * 16; rr += step) {
        const int g = group_of(tile0, rr >> 4);
        const int pos = rr - tile0[g] * 16;
        int src = -1, dst = -1;
        if (pos < begin[g + 1] - begin[g]) {
            if (g < ng_routed) {
                const int e = begin[g] + pos;
                src = entry_token[e];
                dst = src * slots + entry_k[e];
                if (src_per_slot) src = dst;  // the activations come per (token, slot) as well
            } else {
                src = pos;
                dst = pos * slots + sh_slot;
            }
        }
        row_src[rr] = src, out_row[rr] = dst;
    }
}

// Grouping of given ids and the plan above in one launch, a workgroup per expert (the last one stands for the shared expert): each
// counts the pairs of every expert in LDS -- the ids are a few KB that the L2 hands out --, adds up what lies ahead of its own
// expert, and places its own pairs in the order of the ids, so a repeated (token, expert) needs no case of its own.  The lists, the
// plan and the quantizing workgroups are those of build_groups_kernel and moe_gemm_plan_kernel, which took two launches and
// sixteen workgroups that placed every expert's pairs by bit masks over the tokens.
// Latency: one read of the ids, LDS counters, two barriers, the scattered stores.  256 + 1 experts, top-8, 2048 x 512: at 1500 tokens 10.5 + 6.8
// -> 12.2 us by trace, the block at 256 135.1 -> 132.6; 64 experts, top-6, at 192 / 256 tokens 66.0 / 64.5 ->
// 59.7 / 59.5, 16 experts, top-2, 1024 x 256 at 400 / 700 tokens 52.7 / 59.5 -> 43.8 / 44.9.
__global__ void __launch_bounds__(1024) moe_group_plan_kernel(const int32_t* __restrict__ ids, int n_pairs, int top_k, uint32_t top_k_inverse, int n_experts,
                                                              int32_t* __restrict__ group_expert, int32_t* __restrict__ group_begin,
                                                              int32_t* __restrict__ n_groups, int32_t* __restrict__ entry_token,
                                                              int32_t* __restrict__ entry_k, int slots, int src_per_slot, int sh_tokens,
                                                              int sh_silu_mode, int32_t* __restrict__ plan, int32_t* __restrict__ row_src,
                                                              int32_t* __restrict__ out_row, int mt, int plan_wgs, GroupedRows rows) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if ((int)blockIdx.x >= plan_wgs) {
        quantize_prow_runs(rows, blockIdx.x - (uint32_t)plan_wgs, gridDim.x - (uint32_t)plan_wgs);
        return;
    }
    const int own = blockIdx.x;  // n_experts: the shared expert
    extern __shared__ int32_t plan_sh[];  // pairs of every expert, of this one in every wavefront's run of ids, the sums of wavefront 0
    int32_t* count = plan_sh;
    int32_t* before = count + n_experts;
    int32_t* sums = before + 16;
    // wavefront w holds the pairs [w per, (w + 1) per); bit c of a lane's mine: pair 64 c + lane of them is this expert's
    const int chunks = (n_pairs + 1023) / 1024, first = wave * chunks * 64 + lane;  // chunks <= 64: host-checked
    constexpr int kRound = 16;  // requested together
    int v[kRound];
    auto request = [&](int c0) {
#pragma unroll
        for (int u = 0; u < kRound; ++u) {
            const int i = first + (c0 + u) * 64;
            v[u] = ids[i < n_pairs ? i : n_pairs - 1];
        }
    };
    request(0);
    for (int e = tid; e < n_experts; e += 1024) count[e] = 0;
    __syncthreads();
    uint64_t mine = 0;
    int in_wave = 0;
    for (int c0 = 0; c0 < chunks; c0 += kRound) {
        if (c0 > 0) request(c0);
#pragma unroll
        for (int u = 0; u < kRound; ++u) {
            const bool valid = c0 + u < chunks && first + (c0 + u) * 64 < n_pairs && (uint32_t)v[u] < (uint32_t)n_experts;
            if (valid) atomicAdd(&count[v[u]], 1);
            const bool is_mine = valid && v[u] == own;
            if (is_mine) mine |= (uint64_t)1 << (c0 + u);
            in_wave += __popcll(__ballot(is_mine));
        }
    }
    if (lane == 0) before[wave] = in_wave;
    __syncthreads();
    // what lies ahead of this expert (and, for the totals, of every expert): pairs and tiles, groups and items side by side
    // (at most 2^16 pairs, 2^13 tiles, 2^9 groups)
    const int mt_shift = mt == 2 ? 1 : mt == 4 ? 2 : 3;
    auto ahead_of = [&](int end, int32_t* out) {
        uint32_t pt = 0, gi = 0;
        for (int e = lane; e < end; e += 64) {
            const uint32_t p = (uint32_t)count[e], t = (p + 15) >> 4;
            pt += p | t << 17, gi += (p > 0 ? 1u : 0u) | ((t + mt - 1) >> mt_shift) << 10;
        }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) pt += __shfl_xor(pt, d, 64), gi += __shfl_xor(gi, d, 64);
        if (lane == 0) out[0] = (int)(pt & 0x1ffffu), out[1] = (int)(pt >> 17), out[2] = (int)(gi & 0x3ffu), out[3] = (int)(gi >> 10);
    };
    if (wave == 0) ahead_of(own, sums);
    if (wave == 1 && own == 0) ahead_of(n_experts, sums + 4);
    __syncthreads();
    const int begin = sums[0], tile0 = sums[1], group = sums[2], item0 = sums[3];
    if (own == 0 && tid == 0) {
        const int sh_tiles = (sh_tokens + 15) >> 4, tiles_all = sums[5];
        *n_groups = sums[6], group_begin[sums[6]] = sums[4];
        plan[0] = sums[7] + ((sh_tiles + mt - 1) >> mt_shift), plan[1] = tiles_all + sh_tiles, plan[2] = tiles_all, plan[3] = sh_silu_mode;
    }
    const bool shared = own == n_experts;
    const int here = shared ? sh_tokens : count[own], tiles = (here + 15) >> 4;
    if (here == 0) return;
    if (!shared && tid == 0) group_expert[group] = own, group_begin[group] = begin;
    for (int j = tid; j << mt_shift < tiles; j += 1024) {
        int32_t* item = plan + 4 + 3 * (item0 + j);
        const int t = j << mt_shift;
        item[0] = shared ? -1 : own, item[1] = tile0 + t, item[2] = tiles - t < mt ? tiles - t : mt;
    }
    const int row0 = tile0 * 16;
    for (int p = (shared ? 0 : here) + tid; p < tiles * 16; p += 1024) {  // padding rows, or all of the shared expert's
        row_src[row0 + p] = p < here ? p : -1;
        out_row[row0 + p] = p < here ? p * slots + slots - 1 : -1;
    }
    if (shared) return;
    int at = 0;
    for (int w = 0; w < wave; ++w) at += before[w];
    for (int c = 0; c < chunks; ++c) {
        const bool is_mine = (mine >> c) & 1;
        const uint64_t lanes = __ballot(is_mine);
        if (is_mine) {
            const int pos = at + __popcll(lanes & (((uint64_t)1 << lane) - 1)), i = first + c * 64;
            const int tok = top_k == 1 ? i : (int)__umulhi((uint32_t)i, top_k_inverse), k = i - tok * top_k;
            entry_token[begin + pos] = tok, entry_k[begin + pos] = k;
            const int dst = tok * slots + k;
            row_src[row0 + pos] = src_per_slot ? dst : tok, out_row[row0 + pos] = dst;
        }
        at += __popcll(lanes);
    }
}

}  // namespace

// upper bounds: `entries` counts every row of the plan (the routed pairs and, with a shared expert, every token once
// more), groups_max every group (the experts, + 1 with a shared expert)
int64_t moe_gemm_tiles_max(int64_t entries, int64_t groups_max) { return (entries + 15) / 16 + groups_max; }
// (sized for the smallest items a plan may be cut into, so that the lists behind the items lie at one place whatever
// the item size of a launch)
int64_t moe_gemm_items_max(int64_t entries, int64_t groups_max) {  // a multiple of four: the row arrays behind the items stay 16-byte aligned
    return ((entries + 16 * kMTilesSmall - 1) / (16 * kMTilesSmall) + groups_max + 3) & ~(int64_t)3;
}
// ... of a launch whose items hold up to mt tiles: a group of r rows has at most r / (16 mt) + 1
static int64_t moe_gemm_items_of(int64_t entries, int64_t groups_max, int mt) { return (entries + 16 * mt - 1) / (16 * mt) + groups_max; }
size_t moe_gemm_plan_ints(int64_t entries, int64_t groups_max) {
    return 4 + 3 * (size_t)moe_gemm_items_max(entries, groups_max) + 2 * 16 * (size_t)moe_gemm_tiles_max(entries, groups_max);
}

// The grouping of the given ids and the plan over it.  One launch up to kGroupPlanExperts experts (a workgroup each, two to a compute
// unit: all at once) and 64 x 1024 pairs (a lane's bits); beyond, two launches as before.
constexpr int64_t kGroupPlanExperts = 512, kGroupPlanPairs = 64 * 1024;
hipError_t launch_moe_group_plan(const int32_t* ids, int64_t n, int top_k, int64_t n_experts, int32_t* group_expert, int32_t* group_begin,
                                 int32_t* n_groups, int32_t* entry_token, int32_t* entry_k, int slots, bool src_per_slot, int64_t sh_tokens,
                                 int sh_silu_mode, int32_t* plan, hipStream_t stream, int mt, const GroupedRows& rows) {
    const int64_t entries = n * top_k + sh_tokens, groups_max = n_experts + (sh_tokens > 0 ? 1 : 0);
    // (a grid holds fewer than 2^32 threads, four million workgroups of 1024: beyond kQuantWgs a workgroup takes several runs of rows)
    constexpr int64_t kQuantWgs = 1 << 16;
    const int64_t quant_runs = rows.x ? (rows.n + 15) / 16 * rows.nb : 0, quant_wgs = quant_runs < kQuantWgs ? quant_runs : kQuantWgs;
    if (quant_runs >= (int64_t)1 << 31 || (rows.x && (rows.nb > 65535 || rows.n >= (int64_t)1 << 31))) return hipErrorInvalidValue;
    if (groups_max > 4097 || (mt != kMTilesSmall && mt != kMTilesMid && mt != kMTilesPerGroup)) return hipErrorInvalidValue;
    if (entries == 0) return hipSuccess;
    int32_t* row_src = plan + 4 + 3 * moe_gemm_items_max(entries, groups_max);
    int32_t* out_row = row_src + 16 * moe_gemm_tiles_max(entries, groups_max);
    if (n_experts <= kGroupPlanExperts && n * top_k <= kGroupPlanPairs) {
        MQ_LAUNCH(moe_group_plan_kernel, dim3((unsigned)(groups_max + quant_wgs)), dim3(1024), (size_t)(n_experts + 24) * sizeof(int32_t), stream, ids,
                  (int)(n * top_k), top_k, (uint32_t)((((uint64_t)1 << 32) + top_k - 1) / top_k), (int)n_experts, group_expert, group_begin, n_groups, entry_token, entry_k, slots, src_per_slot ? 1 : 0,
                  (int)sh_tokens, sh_silu_mode, plan, row_src, out_row, mt, (int)groups_max, rows);
        return hipGetLastError();
    }
    if (hipError_t e = launch_build_groups(ids, n, top_k, n_experts, group_expert, group_begin, n_groups, entry_token, entry_k, stream); e != hipSuccess) return e;
    const int64_t rows_max = 16 * moe_gemm_tiles_max(entries, groups_max);
    const unsigned wgs = (unsigned)(rows_max / 1024 < 1 ? 1 : (rows_max / 1024 > 64 ? 64 : rows_max / 1024));
    MQ_LAUNCH(moe_gemm_plan_kernel, dim3(wgs + (unsigned)quant_wgs), dim3(1024), 3 * (size_t)(groups_max + 2) * sizeof(int32_t), stream, n_groups,
                       group_expert, group_begin, entry_token, entry_k, slots, src_per_slot ? 1 : 0, (int)groups_max, (int)sh_tokens,
                       slots - 1, sh_silu_mode, plan, row_src, out_row, mt, (int)wgs, rows);
    return hipGetLastError();
}

// Rows of the plan's tiles in the P-major layout: gathered from x by the plan's row list (swiglu == false; x_in_place: by its list of
// output rows, x being what an expert-grouped launch scattered), or
// silu(gate) * up of two planes that already are in the plan's row order (swiglu == true; h_out, if given, receives
// those rows as fp32 at their per-(token, slot) places).
hipError_t launch_quantize_q8k_pmajor_grouped(const float* x, const float* x2, bool swiglu, int silu_mode, int64_t ldx, int64_t k,
                                              int64_t entries, int64_t groups_max, const int32_t* plan, uint8_t* ap, float* h_out,
                                              int64_t ldh, hipStream_t stream, bool x_in_place) {
    const int64_t nb = k / kQK, m_tiles = moe_gemm_tiles_max(entries, groups_max);
    if (m_tiles == 0 || nb == 0) return hipSuccess;
    if (nb > 65535 || m_tiles >= (int64_t)1 << 31) return hipErrorInvalidValue;
    const int32_t* row_src = plan + 4 + 3 * moe_gemm_items_max(entries, groups_max);
    if (swiglu) {
        MQ_LAUNCH(quantize_q8k_pmajor_kernel<true>, dim3((unsigned)m_tiles, (unsigned)nb), dim3(256), 0, stream, x, x2, silu_mode,
                           h_out, ldh, m_tiles * 16, ldx, nb, m_tiles, ap, plan, (const int32_t*)nullptr,
                           row_src + 16 * m_tiles);
    } else {
        MQ_LAUNCH(quantize_q8k_pmajor_kernel<false>, dim3((unsigned)m_tiles, (unsigned)nb), dim3(256), 0, stream, x,
                           (const float*)nullptr, 0, (float*)nullptr, (int64_t)0, m_tiles * 16, ldx, nb, m_tiles, ap, plan,
                           x_in_place ? row_src + 16 * m_tiles : row_src,
                           (const int32_t*)nullptr);
    }
    return hipGetLastError();
}

// y = the plan's tiles . W_expert^T per item.  scatter == false: y [tiles * 16][ldy] in the plan's row order;
// true: row out_row[r] of y (the per-(token, slot) rows of the down product).
int moe_gemm_item_tiles(int64_t entries, int64_t groups) {
    // An expert with more rows than an item takes several items, each of which expands the expert's weights again; an
    // item larger than its expert's rows holds accumulators and LDS for tiles that do not exist, and a compute unit
    // then holds fewer workgroups.  MoE block of 256 + 1 experts, top-8, 2048 x 512, items of 2 / 4 / 8 tiles: 162 / 172 /
    // 209 us at 384 tokens (13 rows per expert), 173 / 181 / 219 at 512, 195 / 203 / 239 at 768, 236 / 224 / 260 at 1024
    // (36 rows), 315 / 276 / 311 at 1536, 385 / 356 / 364 at 2048 (72 rows), 686 / 612 / 615 at 4096.  Swept on Q4_K; the other types take
    // the same items.
    if (groups <= 0) return kMTilesPerGroup;
    return entries <= 30 * groups ? kMTilesSmall : entries <= 160 * groups ? kMTilesMid : kMTilesPerGroup;
}

namespace {
// Two activation buffers are more than the default 64 KB of dynamic LDS: raised once for every form that stages eight tiles.
hipError_t raise_gemm_lds() {
    static bool raised = false;
    if (raised) return hipSuccess;
#define MQ_TILES(KW, WT_, PAIR_, MT_) reinterpret_cast<const void*>(&prefill_gemm_kernel<KW, WT_, PAIR_, MT_, false, true>)
#define MQ_FORM(KW, WT_, PAIR_) MQ_TILES(KW, WT_, PAIR_, 5), MQ_TILES(KW, WT_, PAIR_, 6), MQ_TILES(KW, WT_, PAIR_, 7), MQ_TILES(KW, WT_, PAIR_, 8)
#define MQ_GATHER_FORM(WT_, PAIR_) reinterpret_cast<const void*>(&prefill_gemm_kernel<2, WT_, PAIR_, kMTilesPerGroup, true>)
    for (const void* k : {MQ_FORM(1, kWtQ4, false), MQ_FORM(2, kWtQ4, false), MQ_FORM(2, kWtQ4, true), MQ_FORM(1, kWtQ5, false), MQ_FORM(2, kWtQ5, false),
                          MQ_FORM(2, kWtQ5, true), MQ_FORM(1, kWtQ6, false), MQ_FORM(2, kWtQ6, false), MQ_FORM(2, kWtQ6, true),
                          reinterpret_cast<const void*>(&prefill_gemm_kernel<2, kWtQ4>), reinterpret_cast<const void*>(&prefill_gemm_kernel<2, kWtQ5>),
                          reinterpret_cast<const void*>(&prefill_gemm_kernel<2, kWtQ6>), MQ_GATHER_FORM(kWtQ4, false), MQ_GATHER_FORM(kWtQ5, false), MQ_GATHER_FORM(kWtQ6, false),
                          MQ_GATHER_FORM(kWtQ4, true), MQ_GATHER_FORM(kWtQ5, true), MQ_GATHER_FORM(kWtQ6, true)}) {
        hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * kMTilesPerGroup * kPTileBytes);
        if (e != hipSuccess) return e;
    }
#undef MQ_FORM
#undef MQ_TILES
#undef MQ_GATHER_FORM
    raised = true;
    return hipSuccess;
}
// Where all super-blocks of an item's tiles fit the LDS of four workgroups to a unit (a down product of two super-blocks; of four with
// items of two tiles), a workgroup keeps them and takes this many blocks of 64 rows: MoE block of 256 + 1 experts, top-8, 2048 x 512 at
// 700 / 1500 tokens 165.0 / 240.7 -> 163.4 / 235.0 us.  Shares of the time without, on another card: one block (a single barrier) 0.986 /
// 0.984, two 0.976 / 0.961, four 0.981 / 0.957, eight 1.002 / 0.984 (their last round of workgroups is long); at twice the LDS (two
// workgroups to a unit) 4096 x 1024 at 300 tokens 104 -> 114 us.
constexpr int kResidentTiles = 8, kResidentRowBlocks = 2;
constexpr int64_t kGatherMaxRows = ((int64_t)1 << 31) / kPRowBytes;  // a row's offset in its plane is a 32-bit one
int pace_of(int wtype) { return wtype == kTypeQ6K ? 2 : wtype == kTypeQ5K ? 1 : 0; }
bool gemm_type(int wtype) { return wtype == kTypeQ4K || wtype == kTypeQ5K || wtype == kTypeQ6K; }
// GO(form constant) for the weight type of a launch
#define MQ_BY_TYPE(wtype, GO)              \
    do {                                   \
        if ((wtype) == kTypeQ6K) GO(kWtQ6); \
        else if ((wtype) == kTypeQ5K) GO(kWtQ5); \
        else GO(kWtQ4);                    \
    } while (0)
// LDS of a dense GEMM's workgroup, whatever its tiles: two to a compute unit, as the estimate of a shape has it.  With as many as fit, 448
// workgroups of fewer tiles come to lie three to a unit beside units with one (Q6_K 14336 x 4096 at 200 rows 41.8 -> 46.1 us).
constexpr size_t kGemmLds = 2 * kMTilesPerGroup * kPTileBytes;
// GO(type, activation tiles of the form): five to eight tiles of a workgroup in a form of their own, fewer in that of five
#define MQ_BY_COUNT(tiles, GO, WT_)        \
    do {                                   \
        if ((tiles) >= 8) GO(WT_, 8);      \
        else if ((tiles) == 7) GO(WT_, 7); \
        else if ((tiles) == 6) GO(WT_, 6); \
        else GO(WT_, 5);                   \
    } while (0)
}  // namespace

hipError_t launch_prefill_gemm_grouped(const uint8_t* w, int wtype, int64_t expert_bytes, const uint8_t* w_shared, int64_t rows,
                                       int64_t nb, const uint8_t* ap, int64_t gathered, int64_t entries, int64_t groups_max, const int32_t* plan,
                                       bool scatter, float* y, int64_t ldy, hipStream_t stream, int mt) {
    if (!gemm_type(wtype)) return hipErrorInvalidValue;
    if (mt != kMTilesSmall && mt != kMTilesMid && mt != kMTilesPerGroup) return hipErrorInvalidValue;
    const int64_t rowtiles = (rows + 15) / 16, m_tiles = moe_gemm_tiles_max(entries, groups_max);
    const int64_t items = moe_gemm_items_max(entries, groups_max);
    if (rowtiles == 0 || items == 0) return hipSuccess;
    if (items > 65535 || gathered > kGatherMaxRows) return hipErrorInvalidValue;
    if (hipError_t e = raise_gemm_lds(); e != hipSuccess) return e;
    const int32_t* row_src = plan + 4 + 3 * items;
    const int32_t* out_row = scatter ? row_src + 16 * m_tiles : nullptr;
    const unsigned live = (unsigned)moe_gemm_items_of(entries, groups_max, mt);
    if (gathered == 0 && mt <= kMTilesMid && nb * mt <= kResidentTiles) {
        const dim3 grid((unsigned)((rowtiles + 4 * kResidentRowBlocks - 1) / (4 * kResidentRowBlocks)), live);
#define MQ_RESIDENT(WT_, MT_)                                                                                                          \
    MQ_LAUNCH((prefill_gemm_resident_kernel<WT_, MT_>), grid, dim3(256), (size_t)nb * MT_ * kPTileBytes + MT_ * 64, stream, w, (int)rowtiles, rows, (int)nb, ap, \
              m_tiles, y, ldy, plan, expert_bytes, out_row, w_shared, kResidentRowBlocks)
#define MQ_GO(WT_)                                       \
    if (mt == kMTilesSmall) MQ_RESIDENT(WT_, kMTilesSmall); \
    else MQ_RESIDENT(WT_, kMTilesMid)
        MQ_BY_TYPE(wtype, MQ_GO);
#undef MQ_GO
#undef MQ_RESIDENT
        return hipGetLastError();
    }
    const dim3 narrow((unsigned)((rowtiles + 3) / 4), live), wide((unsigned)((rowtiles + 7) / 8), live);
#define MQ_GROUPED(KW, WT_, MT_, GATHER_, GRID)                                                                                             \
    MQ_LAUNCH((prefill_gemm_kernel<KW, WT_, false, MT_, GATHER_>), GRID, dim3(256), 2 * MT_ * kPTileBytes, stream, w, rowtiles, rows, nb, ap, \
              m_tiles, m_tiles * 16, y, ldy, (int)nb, (int64_t)0, plan, expert_bytes, out_row, w_shared, (const uint8_t*)nullptr,           \
              (const uint8_t*)nullptr, 0, MT_, row_src, prow_bytes(gathered, 1))
    // two and four tiles: one weight tile per wavefront -- few registers, several workgroups to a compute unit
#define MQ_BY_TILES(WT_, GATHER_)                                                 \
    if (mt == kMTilesSmall) MQ_GROUPED(1, WT_, kMTilesSmall, GATHER_, narrow);    \
    else if (mt == kMTilesMid) MQ_GROUPED(1, WT_, kMTilesMid, GATHER_, narrow);   \
    else MQ_GROUPED(2, WT_, kMTilesPerGroup, GATHER_, wide)
#define MQ_GO(WT_)                                  \
    do {                                            \
        if (gathered > 0) { MQ_BY_TILES(WT_, true); } \
        else { MQ_BY_TILES(WT_, false); }           \
    } while (0)
    MQ_BY_TYPE(wtype, MQ_GO);
#undef MQ_GO
#undef MQ_BY_TILES
#undef MQ_GROUPED
    return hipGetLastError();
}

GemmShape gemm_shape(int wtype, int64_t rows, int64_t nb, int64_t n) { return choose_shape(kPace[pace_of(wtype)], false, rows, nb, n); }

// Rows that do not divide by four have no runs of their own; the launch runs over the rows padded to four instead (the same row tiles) where
// that shape is the shorter one, and the planes' sum leaves the padding out.  Without it every workgroup of a short matrix walks all of
// K: 128 products of ragged matrices (512 to 16,384 rows, 1024 to 14,080 columns, 17 to 2048 tokens) take 0.826 of the time with it, with the
// operands read ahead; Q5_K 791 x 13312 at 221 tokens 72.9 -> 27.1 us, Q6_K 1107 x 8448 at 51 tokens 35.8 -> 16.6.
GemmShape gemm_launch_shape(int wtype, int64_t rows, int64_t nb, int64_t n) {
    const GemmShape own = gemm_shape(wtype, rows, nb, n);
    if ((rows & 3) == 0) return own;
    const GemmShape padded = gemm_shape(wtype, plane_pitch(rows), nb, n);
    return padded.us < own.us ? padded : own;
}

// The pair form: h[tok][row] = silu(gate[row] . x[tok]) * (up[row] . x[tok]).  It has no K split (SiLU is not linear): for a few rows of
// a long K two launches with K in runs and the SwiGLU pass over their planes are faster, by up to half (1 to 4 % of the fitted
// pairs); taken where the estimate, with 8 us of quantizer on both sides, says so by 6 % (then never slower by more than 5 %).
// In an FFN (then_quantized) the SwiGLU pass of two launches is the down product's quantizer, which the pair form adds: 4 us and
// more, compared as it is.  Of 7,650 random FFNs (17 to 1200 rows) the pair lost over 2 % on 89 without that, up to 9 % (Q5_K
// 4608 -> 10496 at 17 rows 61.0 against 56.0 us); with it the choice does on 15 of 7,490, at most 7 %.
bool gemm_pair_shape(int wtype, int64_t rows, int64_t nb, int64_t n, bool then_quantized, GemmShape* shape) {
    if (!gemm_type(wtype) || rows <= 0 || n <= 0) return false;
    *shape = choose_shape(kPace[pace_of(wtype)], true, rows, nb, n);
    const float out = 1e-6f * (float)(n * rows), one_launch = shape->us + 0.25f * out + 8.0f;
    const float two_launches = 2.0f * gemm_launch_shape(wtype, rows, nb, n).us + 8.5f + 3.15f * out + 8.0f;
    return two_launches >= (then_quantized ? one_launch + 4.0f + 0.82f * out : 0.94f * one_launch);
}

hipError_t launch_prefill_gemm_pair(const uint8_t* gate, const uint8_t* up, int wtype, int64_t rows, int64_t nb, const uint8_t* ap,
                                    int64_t n, int silu_mode, float* h, int64_t ldh, const GemmShape& ps, hipStream_t stream) {
    const int64_t rowtiles = (rows + 15) / 16, m_tiles = (n + 15) / 16;
    if (rowtiles == 0 || m_tiles == 0) return hipSuccess;
    if (!gemm_type(wtype) || ps.splits != 1 || ps.groups > 65535u) return hipErrorInvalidValue;
    if (hipError_t e = raise_gemm_lds(); e != hipSuccess) return e;
#define MQ_PAIR(WT_, MT_)                                                                                                                 \
    MQ_LAUNCH((prefill_gemm_kernel<2, WT_, true, MT_, false, true>), dim3(ps.row_wgs, ps.groups, 1u), dim3(256), kGemmLds, stream, \
              gate, rowtiles, rows, nb, ap, m_tiles, n, h, ldh, (int)nb, (int64_t)0, (const int32_t*)nullptr, (int64_t)0,               \
              (const int32_t*)nullptr, (const uint8_t*)nullptr, up, (const uint8_t*)nullptr, silu_mode, ps.tiles_per_wg)
#define MQ_GO(WT_) MQ_BY_COUNT(ps.tiles_per_wg, MQ_PAIR, WT_)
    MQ_BY_TYPE(wtype, MQ_GO);
#undef MQ_GO
#undef MQ_PAIR
    return hipGetLastError();
}

// The expert-grouped pair form: scatter == false: h [tiles * 16][ldh] in the plan's row order; true: row out_row[r] of h.
hipError_t launch_prefill_gemm_grouped_pair(const uint8_t* gate, const uint8_t* up, int wtype, int64_t expert_bytes,
                                            const uint8_t* gate_shared, const uint8_t* up_shared, int64_t rows, int64_t nb,
                                            const uint8_t* a_rows, int64_t gathered, int64_t entries, int64_t groups_max, const int32_t* plan, bool scatter,
                                            int silu_mode, float* h, int64_t ldh, hipStream_t stream, int mt) {
    if (!gemm_type(wtype) || (mt != kMTilesSmall && mt != kMTilesMid && mt != kMTilesPerGroup)) return hipErrorInvalidValue;
    const int64_t rowtiles = (rows + 15) / 16, m_tiles = moe_gemm_tiles_max(entries, groups_max);
    const int64_t items = moe_gemm_items_max(entries, groups_max);
    if (rowtiles == 0 || items == 0) return hipSuccess;
    if (items > 65535 || gathered < 1 || gathered > kGatherMaxRows) return hipErrorInvalidValue;
    if (hipError_t e = raise_gemm_lds(); e != hipSuccess) return e;
    const int32_t* row_src = plan + 4 + 3 * items;
    const int32_t* out_row = scatter ? row_src + 16 * m_tiles : nullptr;
    const dim3 grid((unsigned)((rowtiles + 3) / 4), (unsigned)moe_gemm_items_of(entries, groups_max, mt));
#define MQ_GROUPED(WT_, MT_)                                                                                                                     \
    MQ_LAUNCH((prefill_gemm_kernel<2, WT_, true, MT_, true>), grid, dim3(256), 2 * MT_ * kPTileBytes, stream, gate, rowtiles, rows, nb, a_rows, m_tiles, \
              m_tiles * 16, h, ldh, (int)nb, (int64_t)0, plan, expert_bytes, out_row, gate_shared, up, up_shared, silu_mode, MT_, row_src, prow_bytes(gathered, 1))
#define MQ_GO(WT_)                                           \
    if (mt == kMTilesSmall) MQ_GROUPED(WT_, kMTilesSmall);   \
    else if (mt == kMTilesMid) MQ_GROUPED(WT_, kMTilesMid);  \
    else MQ_GROUPED(WT_, kMTilesPerGroup)
    MQ_BY_TYPE(wtype, MQ_GO);
#undef MQ_GO
#undef MQ_GROUPED
    return hipGetLastError();
}

size_t gemm_part_bytes(const GemmShape& ps, int64_t rows, int64_t n) {
    return ps.splits > 1 ? planes_bytes(ps.splits, rows, n) : 0;
}

size_t prow_bytes(int64_t n, int64_t nb) { return (size_t)n * (size_t)nb * kPRowBytes; }

size_t pmajor_bytes(int64_t n, int64_t nb) { return (size_t)((n + 15) / 16) * (size_t)nb * kPTileBytes; }

hipError_t launch_quantize_q8k_pmajor(const float* x, int64_t n, int64_t ldx, int64_t k, uint8_t* ap,
                                      hipStream_t stream, const int32_t* plan) {
    const int64_t nb = k / kQK, m_tiles = (n + 15) / 16;
    if (m_tiles == 0 || nb == 0) return hipSuccess;
    if (nb > 65535 || m_tiles >= (int64_t)1 << 31) return hipErrorInvalidValue;
    if (m_tiles * nb <= 64 && !plan) {  // a few workgroups (sixteen rows of a decode-width product): a wavefront per row
        MQ_LAUNCH((quantize_q8k_pmajor_kernel<false, 1>), dim3((unsigned)m_tiles, (unsigned)nb), dim3(1024), 0, stream, x,
                  (const float*)nullptr, 0, (float*)nullptr, (int64_t)0, n, ldx, nb, m_tiles, ap, plan, (const int32_t*)nullptr,
                  (const int32_t*)nullptr);
        return hipGetLastError();
    }
    MQ_LAUNCH(quantize_q8k_pmajor_kernel<false>, dim3((unsigned)m_tiles, (unsigned)nb), dim3(256), 0, stream, x,
                       (const float*)nullptr, 0, (float*)nullptr, (int64_t)0, n, ldx, nb, m_tiles, ap, plan,
                       (const int32_t*)nullptr, (const int32_t*)nullptr);
    return hipGetLastError();
}

hipError_t launch_swiglu_quantize_q8k_pmajor(const float* gate, const float* up, int64_t n, int64_t ldx, int64_t k,
                                             int silu_mode, float* h_out, int64_t ldh, uint8_t* ap, hipStream_t stream) {
    const int64_t nb = k / kQK, m_tiles = (n + 15) / 16;
    if (m_tiles == 0 || nb == 0) return hipSuccess;
    if (nb > 65535 || m_tiles >= (int64_t)1 << 31) return hipErrorInvalidValue;
    MQ_LAUNCH(quantize_q8k_pmajor_kernel<true>, dim3((unsigned)m_tiles, (unsigned)nb), dim3(256), 0, stream, gate, up,
                       silu_mode, h_out, ldh, n, ldx, nb, m_tiles, ap, (const int32_t*)nullptr, (const int32_t*)nullptr,
                       (const int32_t*)nullptr);
    return hipGetLastError();
}

size_t planes_bytes(int splits, int64_t rows, int64_t n) { return (size_t)splits * (size_t)n * (size_t)plane_pitch(rows) * sizeof(float); }

// A run has at least four super-blocks, and one run fewer would leave at most four workgroups to a unit (choose_shape, q80_gemm_runs), each
// of at most 128 rows of outputs by 128: (runs - 1) times the outputs is at most `most`, and so are the outputs of a product in runs.
size_t planes_most(int64_t rows, int64_t nb, int64_t n) {
    const int64_t most = 4 * (int64_t)compute_units() * 128 * 128, outputs = n * plane_pitch(rows);
    if (nb < 8) return 0;
    const int64_t by_units = (outputs < most ? outputs : most) + most;
    return (size_t)(nb / 4 > by_units / outputs ? by_units : nb / 4 * outputs) * sizeof(float);
}

hipError_t launch_sum_planes(const float* part, int splits, int64_t n, int64_t rows, float* y, int64_t ldy, hipStream_t stream) {
    const int64_t pitch = plane_pitch(rows), units = n * (pitch >> 2);
    MQ_LAUNCH(prefill_sum_planes_kernel, dim3((unsigned)((units + 255) / 256)), dim3(256), 0, stream, part, splits, n, rows, pitch, y, ldy);
    return hipGetLastError();
}

hipError_t launch_prefill_gemm(const uint8_t* w, int wtype, int64_t rows, int64_t nb, const uint8_t* ap, int64_t n, float* y,
                               int64_t ldy, float* part, const GemmShape& ps, hipStream_t stream) {
    const int64_t rowtiles = (rows + 15) / 16, m_tiles = (n + 15) / 16;
    if (rowtiles == 0 || m_tiles == 0) return hipSuccess;
    if (!gemm_type(wtype)) return hipErrorInvalidValue;
    if (ps.groups > 65535u) return hipErrorInvalidValue;
    if (ps.splits > 1 && !part) return hipErrorInvalidValue;
    if (hipError_t e = raise_gemm_lds(); e != hipSuccess) return e;
    const bool split = ps.splits > 1;
    float* out = split ? part : y;
    const int64_t ld = split ? plane_pitch(rows) : ldy;
    const int64_t stride = split ? n * ld : 0;
    const dim3 grid(ps.row_wgs, ps.groups, (unsigned)ps.splits);
#define MQ_WIDE(WT_, MT_) MQ_DENSE(2, WT_, MT_)
#define MQ_NARROW(WT_, MT_) MQ_DENSE(1, WT_, MT_)
#define MQ_DENSE(KW, WT_, MT_)                                                                                                            \
    MQ_LAUNCH((prefill_gemm_kernel<KW, WT_, false, MT_, false, true>), grid, dim3(256), kGemmLds, stream, w, rowtiles, rows, nb, ap, m_tiles, \
              n, out, ld, ps.sb_split, stride, (const int32_t*)nullptr, (int64_t)0, (const int32_t*)nullptr, (const uint8_t*)nullptr, \
              (const uint8_t*)nullptr, (const uint8_t*)nullptr, 0, ps.tiles_per_wg)
#define MQ_GO(WT_)                       \
    if (ps.narrow) MQ_BY_COUNT(ps.tiles_per_wg, MQ_NARROW, WT_); \
    else MQ_BY_COUNT(ps.tiles_per_wg, MQ_WIDE, WT_)
    MQ_BY_TYPE(wtype, MQ_GO);
#undef MQ_GO
#undef MQ_NARROW
#undef MQ_WIDE
#undef MQ_DENSE
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    if (split) {
        return launch_sum_planes(part, ps.splits, n, rows, y, ldy, stream);
    }
    return hipGetLastError();
}

}  // namespace mq
