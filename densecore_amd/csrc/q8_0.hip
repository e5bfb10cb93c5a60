// Q8_0 weights x Q8_0 activations at decode widths: y[m][r] = sum_blocks fp16(dx) * fp16(dy) * sum_32 qx * qy.
//
// The reference sends Q8_0 weight matrices (token embeddings used as output head, some attention tensors of
// mixed-precision files) through the same GEMV / small-batch callbacks as the K-quants, with the activations
// quantized to Q8_0 too (core/src/llm/matmul/batched_exec.cpp:630; four-column kernel Q8SmallBatchDot4,
// core/src/llm/matmul/q8_small_batch.h:29-77: per 32-weight block an integer dot and one fused multiply-add with
// fp16(dx) * fp16(dy)).  Here:
//   * quantize_q80_kernel: one wavefront per (row, 256 values): the maximum magnitude of each 32-value block over
//     its eight lanes, d = amax / 127 stored as fp16, codes = round-half-even(x * (127 / amax)) -- ggml's x86
//     quantizer, which lives in a submodule the reference tree does not carry (its parity is unpinned) -- written
//     as the split-slot A operand of common.h (the element order of Q8_K's codes) plus eight fp16 scales per row
//     and 256 values;
//   * q80_matmul_kernel: workgroup = 16 weight rows, its wavefronts split the 256-weight groups of the row and keep
//     a ring of tiles in flight as matmul_kernel does; one K=64 MFMA yields the integer sums of two 32-weight
//     blocks for eight activation rows; acc = fma(dx * dy, float(sum), acc) block by block; partial sums of the
//     wavefronts meet in wave order.  More than eight rows: passes of eight over the same 16 weight rows.
// Integer block sums are exact (mq_debug_block_sums writes them out); fp32 differs from the reference's eight-lane
// order by rounding only.
#include "common.h"
#include "kernels.h"
#include "decode_tile.h"
#include "pmajor.h"

namespace mq {

namespace {

constexpr int kStages = 3;

// The lane's four values of a row (lane l: values 4l .. 4l + 3 of 256) as codes, and the scale of their 32-value block before it is
// rounded to fp16.
__device__ __forceinline__ uint32_t quantize_lane_q80(const float4 v, float& d) {
    const float e[4] = {v.x, v.y, v.z, v.w};
    float local = fmaxf(fmaxf(fabsf(e[0]), fabsf(e[1])), fmaxf(fabsf(e[2]), fabsf(e[3])));
    // largest magnitude of the block = of the eight lanes 8g .. 8g+7 (non-negative floats order like their bits)
    uint32_t a = __float_as_uint(local), t;
    t = dpp_u32<kDppXor1>(a);
    a = t > a ? t : a;
    t = dpp_u32<kDppXor2>(a);
    a = t > a ? t : a;
    t = dpp_u32<kDppHalfMirror>(a);
    a = t > a ? t : a;
    const float amax = __uint_as_float(a);
    d = __fdiv_rn(amax, 127.0f);
    const float id = amax != 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
    uint32_t packed = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) packed |= ((uint32_t)(int)rintf(__fmul_rn(e[j], id)) & 0xffu) << (8 * j);
    return packed;
}

__global__ void __launch_bounds__(256) quantize_q80_kernel(const float* __restrict__ x, int64_t n, int64_t ldx, int64_t nb,
                                                           uint8_t* __restrict__ aq, uint16_t* __restrict__ ah) {
    const int lane = threadIdx.x & 63;
    const int64_t unit = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (unit >= n * nb) return;
    int64_t m, b;
    split_unit(unit, nb, m, b);
    const float4 v = *reinterpret_cast<const float4*>(x + m * ldx + b * kQK + lane * 4);
    float d;
    const uint32_t packed = quantize_lane_q80(v, d);
    // element 4*lane+j: block g = lane/8, index 4*(lane%8)+j; the codes go to the half of the row's slot that
    // belongs to the block's parity, zeros to the other half (the A-major layout of common.h)
    const int g = lane >> 3, h = g & 1, kq = (lane & 7) >> 1;
    const size_t off = aq_offset(m, b, g >> 1, kq, h, nb) + (size_t)(lane & 1) * 4;
    *reinterpret_cast<uint32_t*>(aq + off + h * 8) = packed;
    *reinterpret_cast<uint32_t*>(aq + off + (1 - h) * 8) = 0u;
    if ((lane & 7) == 0) ah[ad_index(m, b, nb) * 8 + g] = __half_as_ushort(__float2half_rn(d));
}

struct Tile80 {
    v4u q[4];  // B operands of the four 64-weight chunks
    v4u sc;    // the eight fp16 d of weight row lane % 16
};
struct A80 {
    v4u q[4];    // split-slot A operand
    v4u s0, s1;  // the eight fp16 d of activation rows 2 kq and 2 kq + 1
};

__device__ __forceinline__ void unpack_halves(const v4u w, float (&out)[8]) {
    const uint32_t words[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        out[2 * i] = half_bits_to_float(words[i] & 0xffffu);
        out[2 * i + 1] = half_bits_to_float(words[i] >> 16);
    }
}

__global__ void __launch_bounds__(512) q80_matmul_kernel(const Q80MatmulArgs p) {
    extern __shared__ float red[];  // [W-1][2][64]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_waves = blockDim.x >> 6;
    const int slot = lane & 15, kq = lane >> 4;
    int64_t rt = blockIdx.x;
    const int nb = (int)p.nb;
    const uint8_t* w = p.w;
    int first = 0, last = (int)p.n;  // activation rows this workgroup multiplies (dense, pairs), or entries of its group
    int g_begin = 0;                 // expert-grouped: first entry of the group (or first token of a shared-expert pass)
    bool g_shared = false;
    const bool grouped = p.group_begin != nullptr;
    if (p.pair_ids) {
        // expert-routed: the grid is flat, workgroup = column g * rowtiles + row tile (a grid's second dimension ends
        // at 65535, a prefill-width block has more pairs); column g is hidden row g = token * slots + slot alone,
        // against the expert that the token's slot names (slots past top_k: the shared expert); rows of dropped
        // pairs are left as they are
        const uint32_t rowtiles = (uint32_t)((p.rows + 15) >> 4);
        const int g = (int)(blockIdx.x / rowtiles), tok = g / p.slots, k = g - tok * p.slots;
        rt = (int64_t)(blockIdx.x - (uint32_t)g * rowtiles);
        if (k < p.top_k) {
            const int e = p.pair_ids[tok * p.top_k + k];
            if (e < 0 || e >= p.n_experts) return;  // the whole workgroup, before any barrier
            w += (size_t)e * p.expert_bytes;
        } else {
            w = p.sh_w;
        }
        first = g;
        last = g + 1;
    } else if (grouped) {
        const int g = blockIdx.y, ng = *p.n_groups;
        const int gi = g < p.max_groups ? g : 0;  // columns of the shared expert read group 0's entries and drop them
        const int g_expert = p.group_expert[gi], b0 = p.group_begin[gi], b1 = p.group_begin[gi + 1];
        if (g < ng) {
            w += (size_t)g_expert * p.expert_bytes;
            g_begin = b0;
            last = b1 - b0;
        } else if (g - ng < (p.sh_tokens + kTokTile - 1) / kTokTile) {
            g_shared = true;
            w = p.sh_w;
            g_begin = (g - ng) * kTokTile;
            last = p.sh_tokens - g_begin < kTokTile ? p.sh_tokens - g_begin : kTokTile;
        } else {
            return;  // the whole workgroup, before any barrier
        }
    }
    // hidden / output row of entry e of the group
    auto group_row = [&](int e) {
        if (g_shared) return (g_begin + e) * p.slots + p.top_k;
        return p.entry_token[g_begin + e] * p.slots + p.entry_k[g_begin + e];
    };
    const uint8_t* tiles = w + tile_offset(rt, 0, nb, kTile80Bytes);
    const int cnt = wave < nb ? (nb - wave + n_waves - 1) / n_waves : 0;  // 256-weight groups wave, wave + W, ...

    for (int chunk = first; chunk < last; chunk += kTokTile) {
        const int count = last - chunk < kTokTile ? last - chunk : kTokTile;
        // a dead slot reads a live row of the pass and stores nothing
        const int a_ent = chunk + ((slot >> 1) < count ? (slot >> 1) : count - 1);
        const int arow = grouped ? group_row(a_ent) : a_ent;
        const size_t a_off = aq_row_offset(arow, nb) + (size_t)kq * 256 + (size_t)(slot & 1) * 16;
        int yrow[2];
        size_t s_off[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const bool live = 2 * kq + j < count;
            const int ent = chunk + (live ? 2 * kq + j : count - 1);
            const int r = grouped ? group_row(ent) : ent;
            yrow[j] = live ? r : -1;
            s_off[j] = ad_index(r, 0, nb) * 8;  // + b * 64 halves per group
        }
        float acc[2] = {0.0f, 0.0f};
        if (cnt > 0) {
            Tile80 ring_t[kStages];
            A80 ring_a[kStages];
            auto issue = [&](int st, int i) {
                const int b = i < cnt ? wave + i * n_waves : wave;  // past the end: the first group again, the load count stays fixed
                const uint8_t* tile = tiles + (size_t)b * kTile80Bytes;
#pragma unroll
                for (int c = 0; c < 4; ++c) ring_t[st].q[c] = load_stream16(tile + c * 1024 + lane * 16);
                ring_t[st].sc = load_stream16(tile + kTile80SOff + slot * 16);
#pragma unroll
                for (int c = 0; c < 4; ++c) ring_a[st].q[c] = load16(p.aq + (size_t)b * 4096 + a_off + c * 1024);
                ring_a[st].s0 = load16(p.ah + s_off[0] + (size_t)b * 64);
                ring_a[st].s1 = load16(p.ah + s_off[1] + (size_t)b * 64);
            };
#pragma unroll
            for (int st = 0; st < kStages - 1; ++st) issue(st, st);
            for (int base = 0; base < cnt; base += kStages) {
#pragma unroll
                for (int st = 0; st < kStages; ++st) {
                    const int i = base + st;
                    issue((st + kStages - 1) % kStages, i + kStages - 1);
                    if (i < cnt) {
                        float dx[8], dy[2][8];
                        unpack_halves(ring_t[st].sc, dx);
                        unpack_halves(ring_a[st].s0, dy[0]);
                        unpack_halves(ring_a[st].s1, dy[1]);
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            const v4u av = ring_a[st].q[c], bv = ring_t[st].q[c];
                            const v4i a16 = {(int)av.x, (int)av.y, (int)av.z, (int)av.w};
                            const v4i b16 = {(int)bv.x, (int)bv.y, (int)bv.z, (int)bv.w};
                            const v4i zero = {0, 0, 0, 0};
                            // s[0], s[2]: block 2c of activation rows 2kq and 2kq+1;  s[1], s[3]: block 2c+1
                            const v4i s = __builtin_amdgcn_mfma_i32_16x16x64_i8(a16, b16, zero, 0, 0, 0);
#pragma unroll
                            for (int j = 0; j < 2; ++j)
#pragma unroll
                                for (int h = 0; h < 2; ++h) {
                                    const int k = 2 * c + h;
                                    acc[j] = __fmaf_rn(__fmul_rn(dx[k], dy[j][k]), (float)s[2 * j + h], acc[j]);
                                    if (p.dbg_sum && yrow[j] >= 0 && rt * 16 + slot < p.rows)
                                        p.dbg_sum[(((size_t)(rt * 16 + slot) * (size_t)p.n + (size_t)yrow[j]) * (size_t)nb +
                                                   (size_t)(wave + i * n_waves)) * 8 + k] = s[2 * j + h];
                                }
                        }
                    }
                }
            }
        }
        if (n_waves > 1) {
            if (wave > 0) {
                red[((wave - 1) * 2 + 0) * 64 + lane] = acc[0];
                red[((wave - 1) * 2 + 1) * 64 + lane] = acc[1];
            }
            __syncthreads();
        }
        if (wave == 0) {
            for (int wv = 1; wv < n_waves; ++wv) {
                acc[0] = __fadd_rn(acc[0], red[((wv - 1) * 2 + 0) * 64 + lane]);
                acc[1] = __fadd_rn(acc[1], red[((wv - 1) * 2 + 1) * 64 + lane]);
            }
            const int64_t row = rt * 16 + slot;
            if (row < p.rows) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    if (yrow[j] >= 0) p.y[(size_t)yrow[j] * (size_t)p.ldy + (size_t)row] = acc[j];
            }
        }
        if (n_waves > 1 && chunk + kTokTile < last) __syncthreads();  // red[] is reused by the next pass
    }
}

// ---- more than a few passes of eight: a GEMM -----------------------------------------------------------------------
// Activation tile of sixteen rows x 256 values, 4608 bytes: the codes in the order of a weight tile ([c 0..3][kq][row][16 B]: bytes
// 0..7 of block 2c, elements 8 kq .. +7, then of block 2c + 1), then the block scales as fp32 [8 blocks][16 rows].
constexpr int kQ80ATileBytes = 4096 + 512, kQ80ATileWords = kQ80ATileBytes / 16;

// The quantizer above into these tiles: a workgroup per (tile, 256 values), four rows per wavefront; rows past n are zeros.
__global__ void __launch_bounds__(256) quantize_q80_tiles_kernel(const float* __restrict__ x, int64_t n, int64_t ldx, int64_t m_tiles, uint8_t* __restrict__ ap) {
    __shared__ __align__(16) uint8_t img[kQ80ATileBytes];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t tile = blockIdx.x, b = blockIdx.y;
    float4 v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int64_t m = tile * 16 + wave * 4 + r;
        v[r] = *reinterpret_cast<const float4*>(x + (m < n ? m : n - 1) * ldx + b * kQK + lane * 4);
    }
    const int g = lane >> 3, kq = (lane & 7) >> 1;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int tok = wave * 4 + r;
        const bool live = tile * 16 + tok < n;  // wave-uniform
        float d;
        const uint32_t packed = quantize_lane_q80(v[r], d);
        *reinterpret_cast<uint32_t*>(img + (g >> 1) * 1024 + (kq * 16 + tok) * 16 + (g & 1) * 8 + (lane & 1) * 4) = live ? packed : 0u;
        if ((lane & 7) == 0) *reinterpret_cast<float*>(img + 4096 + (g * 16 + tok) * 4) = live ? __half2float(__float2half_rn(d)) : 0.0f;
    }
    __syncthreads();
    v4u* dst = reinterpret_cast<v4u*>(ap + ((size_t)b * (size_t)m_tiles + (size_t)tile) * kQ80ATileBytes);
    for (int i = tid; i < kQ80ATileWords; i += 256) dst[i] = reinterpret_cast<const v4u*>(img)[i];
}

// A workgroup of four wavefronts: four row tiles x MT activation tiles, the activation tiles of a super-block staged in LDS (double
// buffer, LDS-direct copies a super-block ahead), each wavefront's weight tile in registers, the next one on its way.  One K = 32 MFMA
// forms the sums of a block for sixteen rows of either side; each takes three vector instructions per output, and one more joins a
// super-block's sum, which is what bounds it (100 beside eight MFMAs per tile; twelve LDS reads).  A row's sum is two chains, over
// the even and the odd super-blocks, of chains of eight blocks: against double, the same operands, its error is 0.35 to 0.95 of that of
// the passes of eight, which split a row over one to eight wavefronts (40 products of 2048 to 14336 columns; 4096 columns on eight
// wavefronts 0.82e-7 against 0.92e-7, 14336 1.16e-7 against 1.46e-7).  One chain over the row had up to 2.6 times that error;
// it took 0.97 of the time with one activation tile to a workgroup (154 products of 33 rows and more; at least 0.91, 4096 x 14336 at 64 rows),
// the same with two, 0.995 with four.  Eight chains, one per block of a super-block, are slower yet with one and two tiles (1.010, 1.025).
// The launch of eight-row passes walks all rows
// in one workgroup per row tile: us, passes | this: 8075 x 13312 at 32 / 128 / 500 / 1100 rows 97 / 396 / 1561 / 3438 | 40 / 136 / 206 / 437
// (541 TOP/s), 920 x 6912 26 / 92 / 369 / 811 | 22 / 23 / 27 / 43.
template <int MT>
__global__ void __launch_bounds__(256, 4) q80_gemm_kernel(const uint8_t* __restrict__ w, int64_t rowtiles, int64_t rows, int nb, const uint8_t* __restrict__ ap,
                                                          int64_t m_tiles, int64_t n, float* __restrict__ y, int64_t ldy, int sb_run, int64_t plane) {
    __shared__ __align__(16) uint8_t a_lds[2][MT * kQ80ATileBytes];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, kq = lane >> 4;
    const int64_t mt0 = (int64_t)blockIdx.y * MT;
    const int mt_count = (int)(m_tiles - mt0 < MT ? m_tiles - mt0 : MT);
    const int64_t rt = (int64_t)blockIdx.x * 4 + wave;  // row tiles past the end: the last one again, not stored
    const uint8_t* tile = w + tile_offset(rt < rowtiles ? rt : rowtiles - 1, 0, nb, kTile80Bytes);
    // K in runs over grid.z: super-blocks [begin, end) into plane blockIdx.z
    const int begin = (int)blockIdx.z * sb_run, end = begin + sb_run < nb ? begin + sb_run : nb;
    y += (size_t)blockIdx.z * (size_t)plane;
    float even[MT][4], odd[MT][4];  // sums over the run's even and odd super-blocks
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) even[m][i] = odd[m][i] = 0.0f;
    Tile80 next;
    auto request = [&](int b) {
        request_a_tiles(ap + ((size_t)b * (size_t)m_tiles + (size_t)mt0) * kQ80ATileBytes, a_lds[(b - begin) & 1], mt_count * kQ80ATileWords, wave, lane);
#pragma unroll
        for (int c = 0; c < 4; ++c) next.q[c] = load16(tile + (size_t)b * kTile80Bytes + c * 1024 + lane * 16);
        next.sc = load16(tile + (size_t)b * kTile80Bytes + kTile80SOff + r * 16);
    };
    request(begin);
    auto step = [&](int b, float (&sum)[MT][4]) {
        __builtin_amdgcn_s_waitcnt(0 | (0x7 << 4) | (0xF << 8));  // vmcnt(0): what this thread asked for has landed ...
        __syncthreads();                                          // ... and everybody else's; the other buffer is free
        const Tile80 cur = next;
        if (b + 1 < end) request(b + 1);
        float dx[8];
        unpack_halves(cur.sc, dx);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            if (m < mt_count) {  // uniform over the workgroup
                const uint8_t* at = a_lds[(b - begin) & 1] + m * kQ80ATileBytes;
                float part[4];  // the super-block's sum
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    typedef long v2l __attribute__((ext_vector_type(2)));
                    const v2l av = *reinterpret_cast<const v2l*>(at + c * 1024 + lane * 16), bv = __builtin_bit_cast(v2l, cur.q[c]);
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int k = 2 * c + h;
                        const v4i zero = {0, 0, 0, 0};
                        const v4i s = __builtin_amdgcn_mfma_i32_16x16x32_i8(av[h], bv[h], zero, 0, 0, 0);
                        const float4 dy = *reinterpret_cast<const float4*>(at + 4096 + (k * 16 + kq * 4) * 4);
                        const float dyv[4] = {dy.x, dy.y, dy.z, dy.w};
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float d = __fmul_rn(dx[k], dyv[i]);
                            part[i] = k == 0 ? __fmul_rn(d, (float)s[i]) : __fmaf_rn(d, (float)s[i], part[i]);
                        }
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) sum[m][i] = __fadd_rn(sum[m][i], part[i]);
            }
        }
    };
    int b = begin;
    for (; b + 1 < end; b += 2) {
        step(b, even);
        step(b + 1, odd);
    }
    if (b < end) step(b, even);
    const int64_t row = rt * 16 + r;
    if (rt >= rowtiles || row >= rows) return;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t tok = (mt0 + m) * 16 + kq * 4 + i;
            if (tok < n) y[tok * ldy + row] = __fadd_rn(even[m][i], odd[m][i]);
        }
}

}  // namespace

// Activation tiles to a workgroup: as many as leave two workgroups for every unit
int q80_gemm_tiles(int64_t rows, int64_t n) {
    const int64_t row_wgs = ((rows + 15) / 16 + 3) / 4, m_tiles = (n + 15) / 16, enough = 2 * (int64_t)compute_units();
    // (no more than there are: the form of four holds two workgroups fewer to a unit)
    return m_tiles > 2 && row_wgs * ((m_tiles + 3) / 4) >= enough ? 4 : m_tiles > 1 && row_wgs * ((m_tiles + 1) / 2) >= enough ? 2 : 1;
}

// K in runs of at least four super-blocks where the estimate of the GEMM (api.hip) for a run, with a launch and the planes written and read,
// is under 0.9 of that of K whole: a workgroup walks its super-blocks one after the other, half a microsecond each, whatever units that
// leaves idle.  us before | after: 527 x 12544 at 148 rows 39.0 | 20.2, 1866 x 10240 at 27 31.3 | 16.0, 1140 x 13056 at 61 39.4 | 19.4,
// 6315 x 6912 at 15 23.0 | 15.6, 5903 x 12544 at 28 38.4 | 31.1; 137 products 0.949 of the time, those left whole 1.000.
int q80_gemm_runs(int64_t rows, int64_t nb, int64_t n) {
    const int64_t m_tiles = (n + 15) / 16, mt = q80_gemm_tiles(rows, n), wgs = ((rows + 15) / 16 + 3) / 4 * ((m_tiles + mt - 1) / mt);
    float best = 0.0f;
    int runs = 1;
    for (int s = 1; s <= 16 && (s == 1 || nb >= 4 * s); ++s) {
        const int64_t sb = (nb + s - 1) / s;
        if ((nb + sb - 1) / sb != s) continue;  // a count that leaves no empty run
        const float load = (float)(wgs * s) / (float)(2 * compute_units()), k = (float)sb;
        float us = 6.8f + 0.51f * k + (load > 1.0f ? 1.18f * k * (float)mt * (load - 1.0f) : 0.0f) + 19e-6f * (float)rows * (float)nb;
        if (s > 1) us += 2.8f + 0.55e-6f * (float)s * (float)(n * rows);
        if (s == 1 || us < best) best = s == 1 ? 0.9f * us : us, runs = s;
        if (load > 2.0f) break;  // two rounds: further runs only add planes
    }
    return runs;
}

size_t q80_tiles_bytes(int64_t n, int64_t nb) { return (size_t)((n + 15) / 16) * (size_t)nb * kQ80ATileBytes; }

hipError_t launch_q80_gemm(const uint8_t* w, int64_t rows, int64_t nb, const float* x, int64_t n, int64_t ldx, uint8_t* ap, float* y, int64_t ldy, float* part,
                           int runs, hipStream_t stream) {
    const int64_t rowtiles = (rows + 15) / 16, m_tiles = (n + 15) / 16, row_wgs = (rowtiles + 3) / 4;
    if (rows <= 0 || nb <= 0 || n <= 0 || !w || !x || !ap || !y || ldy < rows || ldx < nb * kQK) return hipErrorInvalidValue;
    if (nb > 65535 || m_tiles > 65535 || (ldx & 3) || (reinterpret_cast<uintptr_t>(x) & 15u)) return hipErrorInvalidValue;
    MQ_LAUNCH(quantize_q80_tiles_kernel, dim3((unsigned)m_tiles, (unsigned)nb), dim3(256), 0, stream, x, n, ldx, m_tiles, ap);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    const int tiles = q80_gemm_tiles(rows, n), sb_run = (int)((nb + runs - 1) / runs);
    if (runs < 1 || (runs > 1 && !part)) return hipErrorInvalidValue;
    float* out = runs > 1 ? part : y;
    const int64_t ld = runs > 1 ? plane_pitch(rows) : ldy, plane = runs > 1 ? n * ld : 0;
#define MQ_Q80(MT)                                                                                                                     \
    MQ_LAUNCH(q80_gemm_kernel<MT>, dim3((unsigned)row_wgs, (unsigned)((m_tiles + MT - 1) / MT), (unsigned)runs), dim3(256), 0, stream, w, rowtiles, rows, (int)nb, \
              (const uint8_t*)ap, m_tiles, n, out, ld, sb_run, plane)
    if (tiles == 4) MQ_Q80(4);
    else if (tiles == 2) MQ_Q80(2);
    else MQ_Q80(1);
#undef MQ_Q80
    if (hipError_t e = hipGetLastError(); e != hipSuccess || runs == 1) return e;
    return launch_sum_planes(part, runs, n, rows, y, ldy, stream);
}

size_t q80_scale_bytes(int64_t n, int64_t nb) { return ad_count(n, nb) * 8 * sizeof(uint16_t); }

hipError_t launch_quantize_q80(const float* x, int64_t n, int64_t ldx, int64_t cols, uint8_t* aq, uint16_t* ah, hipStream_t stream) {
    const int64_t nb = cols / kQK, units = n * nb;
    if (units == 0) return hipSuccess;
    if (units >= (int64_t)1 << 31) return hipErrorInvalidValue;  // split_unit divides in 32 bits
    if ((cols % kQK) || ldx < cols || (ldx & 3) || (reinterpret_cast<uintptr_t>(x) & 15u)) return hipErrorInvalidValue;
    MQ_LAUNCH(quantize_q80_kernel, dim3((unsigned)((units + 3) / 4)), dim3(256), 0, stream, x, n, ldx, nb, aq, ah);
    return hipGetLastError();
}

hipError_t launch_q80_matmul(const Q80MatmulArgs& a, hipStream_t stream) {
    if (a.rows <= 0 || a.nb <= 0 || a.n <= 0 || !a.w || !a.aq || !a.ah || !a.y || a.ldy < a.rows) return hipErrorInvalidValue;
    const bool grouped = a.group_begin != nullptr;
    if ((a.pair_ids || grouped) && (a.top_k <= 0 || a.slots < a.top_k || a.n % a.slots || a.dbg_sum || (a.slots > a.top_k && !a.sh_w)))
        return hipErrorInvalidValue;
    if (grouped && (a.pair_ids || !a.group_expert || !a.n_groups || !a.entry_token || !a.entry_k || a.max_groups <= 0)) return hipErrorInvalidValue;
    const int64_t rowtiles = (a.rows + 15) / 16;
    if (grouped) {
        const int64_t columns = (int64_t)a.max_groups + (a.sh_tokens + kTokTile - 1) / kTokTile;
        if (columns > 65535) return hipErrorInvalidValue;
        const int waves = pick_waves(a.nb, rowtiles * columns);
        MQ_LAUNCH(q80_matmul_kernel, dim3((unsigned)rowtiles, (unsigned)columns), dim3(64 * waves),
                           waves > 1 ? (size_t)(waves - 1) * 2 * 64 * sizeof(float) : 0, stream, a);
        return hipGetLastError();
    }
    const int64_t columns = a.pair_ids ? a.n : 1;
    if (rowtiles * columns >= (int64_t)1 << 31) return hipErrorInvalidValue;
    const int waves = pick_waves(a.nb, rowtiles * columns);
    MQ_LAUNCH(q80_matmul_kernel, dim3((unsigned)(rowtiles * columns)), dim3(64 * waves),
                       waves > 1 ? (size_t)(waves - 1) * 2 * 64 * sizeof(float) : 0, stream, a);
    return hipGetLastError();
}

}  // namespace mq
