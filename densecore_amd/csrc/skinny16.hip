// Dense products of nine to 64 activation rows: the rows as one to four activation tiles of sixteen per streamed weight tile.
#include <hip/hip_ext.h>

#include "common.h"
#include "kernels.h"
#include "decode_tile.h"
#include "pmajor.h"
#include "weight_digits.h"

namespace mq {

namespace {

// ---- nine to 64 activation rows against a streamed matrix ------------------------------------------------
// The decode kernels multiply a weight tile with EIGHT activation rows per MFMA (the sixteen operand rows hold a row's
// two sub-blocks of a 64-weight chunk side by side, the sub-block scales are applied on the vector unit); from nine rows
// they take two such token tiles per weight tile: 16 MFMAs and ~147 vector instructions.  This kernel multiplies the
// same rows as ONE tile of sixteen, the way prefill_gemm_kernel does (scale digits folded into the weight operand, the
// min term as one fp16 MFMA): 9 MFMAs and ~126 vector instructions per weight tile.  Everything else is
// dense_lds_kernel's (dense_lds.hip): eight wavefronts, WPR of them per row tile taking the super-blocks h, h + WPR, ...
// in ascending order, partial sums met in wave order, two register stages of raw weight tiles; the rows' quantized
// activations -- here P-major tiles -- are staged in LDS once per workgroup while the first weight tiles travel, or,
// where all super-blocks do not fit LDS (GA: the 14336 columns of an FFN's down projection), requested from global
// memory a stage ahead, beside the weight tile (six loads, all answered by the L2).  The integers of a (row, token,
// super-block) are the same and so is the fp32 update, (wd * yd) * dot - (wm * yd) * min_dot added to the running
// sum: the same bits as dense_lds_kernel and matmul_kernel.
// WT: the weight tile as two chains of byte digits whatever its type (weight_digits.h; Q5_K with one or two activation tiles as
// two and a chain for the fifth code bits), the decode kernels' integers and their update.  Q6_K as digits takes eight MFMAs
// per activation tile in place of sixteen over the bytes of one scale group each with the group sums scaled on the vector
// unit: an FFN of 4096 -> 14336 -> 4096 all Q6_K at 30 rows 56.3 -> 48.7 us, with a Q6_K down projection at 40 rows 56.8 -> 50.6.
// LDS: [nb][4688] activation tiles (not GA), then the partial sums [8 / WPR][WPR - 1][NMAT][4][64].
// Every wavefront has ceil(nb / WPR) stages; FLOW 1: that count is odd (a single run); 0: even, a single run or runs of an even number
// of stages; 2: even, runs of an odd number of stages.  Where nb % WPR != 0 (a single run; the split that dense_waves gives all decode
// kernels for the matrix) the last stage of the wavefronts from nb % WPR on does not exist: they request the last super-block once
// more, another wavefront's at that time, and multiply nothing.  Against a count that divides: 2048 x 5632 at 16 rows (eight wavefronts
// for two) 12.2 -> 8.2 us, 4096 x 11008 at 32 rows (eight for one) 57 -> 15.3.
struct ATile16 {
    v4i a[4];   // the four 64-weight chunks of this lane's operand
    v4f yd;     // the Q8_K scales of rows 4 kq .. 4 kq + 3
    v8h dg;     // this lane's operand of the min MFMA (fp16 digits of the sub-block sums, or zeros)
};

// (a pair of two tiles read from global memory would spill 46 registers)
constexpr bool skinny16_uneven(int nmat, int wpr, bool ga, int mt) { return wpr > 1 && !(ga && nmat == 2 && mt == 2); }

// MT: activation tiles of sixteen rows (one to four, e.g. two for 17 to 32 rows: the weight tile is expanded once for both, 18
// MFMAs and ~156 vector instructions against the 32 + 294 of two passes over two token tiles of eight each).  With two
// tiles the partial sums share LDS with the activation tiles (one more barrier before they are written).
template <int NMAT, int WPR, int FLOW, bool GA, int MT, int WT = kWtQ4>
__global__ void __launch_bounds__(512) skinny16_kernel(const Skinny16Args p) {
    constexpr bool ODD = FLOW == 1;  // (FLOW: the shape of the stage loop, below)
    constexpr int RPW = 8 / WPR;  // row tiles per workgroup
    constexpr bool Q5 = WT == kWtQ5, Q6 = WT == kWtQ6;
    constexpr int kStride = tile_stride<WT>();
    constexpr int kTileLoads = Q6 ? 5 : Q5 ? 4 : 3;  // requests of a weight tile (load_tile, load_tile6)
    constexpr bool kUneven = skinny16_uneven(NMAT, WPR, GA, MT);
    constexpr bool kRedShares = MT > 1 && !GA;  // the partial sums reuse the activation tiles' LDS
    extern __shared__ __align__(16) uint8_t lds16[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, kq = lane >> 4;
    const int nb = (int)p.nb;
    const int64_t rowtiles = (p.rows + 15) >> 4;
    const int pair = wave / WPR, h = wave % WPR;
    int64_t rt = (int64_t)blockIdx.x * RPW + pair;
    const bool dead = rt >= rowtiles;  // past the last row tile: stream the last one again and store nothing
    if (dead) rt = rowtiles - 1;
    float* red = reinterpret_cast<float*>(lds16 + ((GA || kRedShares) ? (size_t)0 : (size_t)nb * MT * kPTileBytes));  // (one run when the sums lie behind the tiles)

    const uint8_t* tiles[NMAT];
    tiles[0] = p.w0 + tile_offset(rt, 0, nb, kStride);
    if (NMAT == 2) tiles[1] = p.w1 + tile_offset(rt, 0, nb, kStride);
    const int cnt = kUneven ? (nb + WPR - 1) / WPR : nb / WPR;  // stages: super-blocks h, h + WPR, ...
    const bool last_exists = !kUneven || h + (cnt - 1) * WPR < nb;  // wave-uniform

    // lane (r, kq): weight row r of the tile, activation rows 4 kq .. 4 kq + 3 of every activation tile
    const int digit_off = kq < 2 ? kPDigitOff + r * 32 + kq * 16 : kPZeroOff;
    auto read_a = [&](ATile16& t, const uint8_t* at) {
#pragma unroll
        for (int j = 0; j < 4; ++j) t.a[j] = *reinterpret_cast<const v4i*>(at + j * 1024 + lane * 16);
        t.yd = *reinterpret_cast<const v4f*>(at + kPScaleOff + kq * 16);
        if constexpr (!Q6) t.dg = *reinterpret_cast<const v8h*>(at + digit_off);  // (Q6_K has no min term)
    };

    // ---- the activation tiles ([super-block][tile]) -> LDS: a linear copy, 1 KB per request, the wavefronts taking the
    // requests in turn.  Rows too long for LDS in one piece come in `ranges` runs of super-blocks, one run at a time:
    // stage i of every wavefront lies in run i / (cnt / ranges), so the wavefronts change runs together (cnt % ranges == 0,
    // host-checked).
    const int sb_per_range = nb / p.ranges, stages_per_range = cnt / p.ranges;
    auto stage_range = [&](int rg) {
        const uint32_t base = (uint32_t)(uintptr_t)(lds_ptr_t)lds16;
        const int words = sb_per_range * MT * kPTileWords;
        const uint8_t* src = p.ap + (size_t)rg * (size_t)words * 16;
        for (int c = wave; c * 64 < words; c += 8) {
            const int first = c * 64;
            if (first + lane < words) {
                const uint8_t* g = src + (size_t)(first + lane) * 16;
                const uint32_t dst = base + (uint32_t)first * 16u;
                lds_direct<16>(g, dst);
            }
        }
    };
    if constexpr (!GA) stage_range(0);

    typename TileOf<WT>::Regs ring_t[2][NMAT];
    ATile16 ring_a[GA ? 2 : 1][GA ? MT : 1];
    auto issue = [&](auto st_c, int i, auto last_c) {  // i < cnt; last_c: i may be cnt - 1 (looking at every request costs Q6_K 2 % and more)
        constexpr int st = decltype(st_c)::value;
        const int b = decltype(last_c)::value && kUneven && h + i * WPR >= nb ? nb - 1 : h + i * WPR;
        if constexpr (GA) {  // ahead of the tiles: they are needed first
#pragma unroll
            for (int t = 0; t < MT; ++t) read_a(ring_a[st][t], p.ap + ((size_t)b * MT + t) * kPTileBytes);
        }
#pragma unroll
        for (int m = 0; m < NMAT; ++m) load_tile_wt<WT>(ring_t[st][m], tiles[m] + (size_t)b * kStride, lane);
    };

    float acc[NMAT][MT][4];
#pragma unroll
    for (int m = 0; m < NMAT; ++m)
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[m][t][i] = 0.0f;

    int b_range0 = 0;  // first super-block of the run in LDS
    auto consume = [&](auto st_c, int i) {
        constexpr int st = decltype(st_c)::value;
        const int b = h + i * WPR;
        const v4i zero = {0, 0, 0, 0};
        const v4f zero_f = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int m = 0; m < NMAT; ++m) {
            // three and four tiles: the second matrix reads the activation tiles from LDS again instead of keeping the first
            // one's copies in registers (they would not fit)
            if (MT > 2 && m > 0) asm volatile("" ::: "memory");
            WTile wt;
            const auto& tr = ring_t[st][m];
            if constexpr (Q6) expand_tile6(tr.ql0, tr.ql1, tr.qh, tr.sc, tr.d, kq, wt);
            else expand_tile<Q5, kFifthChain<WT, MT>>(tr.q0, tr.q1, tr.hdr, Q5 ? tr.qh : v2u{0u, 0u}, kq, wt);
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                ATile16 from_lds;
                if constexpr (!GA) read_a(from_lds, lds16 + ((size_t)(b - b_range0) * MT + t) * kPTileBytes);
                const ATile16& at = GA ? ring_a[GA ? st : 0][GA ? t : 0] : from_lds;
                const float ydv[4] = {at.yd.x, at.yd.y, at.yd.z, at.yd.w};
                v4i hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(at.a[0], wt.hi[0], zero, 0, 0, 0);
                v4i lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(at.a[0], wt.lo[0], zero, 0, 0, 0);
                v4i b5 = zero;
                if constexpr (kFifthChain<WT, MT>) b5 = __builtin_amdgcn_mfma_i32_16x16x64_i8(at.a[0], wt.b5[0], zero, 0, 0, 0);
                v4f mn = zero_f;
                if constexpr (!Q6) mn = __builtin_amdgcn_mfma_f32_16x16x32_f16(at.dg, wt.mins, zero_f, 0, 0, 0);
#pragma unroll
                for (int j = 1; j < 4; ++j) {
                    hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(at.a[j], wt.hi[j], hi, 0, 0, 0);
                    lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(at.a[j], wt.lo[j], lo, 0, 0, 0);
                    if constexpr (kFifthChain<WT, MT>) b5 = __builtin_amdgcn_mfma_i32_16x16x64_i8(at.a[j], wt.b5[j], b5, 0, 0, 0);
                }
#pragma unroll
                for (int i2 = 0; i2 < 4; ++i2) {  // compute_tile's update (decode_tile.h); mn[i2] is the integer min_dot, exactly
                    const int dot = join_digits<WT, MT>(hi[i2], lo[i2], b5[i2]);
                    const float d = __fmul_rn(wt.d, ydv[i2]);
                    if constexpr (Q6) {  // compute_tile6's update (the integers carry a factor 4, d a quarter)
                        acc[m][t][i2] = __fmaf_rn(d, (float)dot, acc[m][t][i2]);
                    } else {
                        const float dm = __fmul_rn(wt.dmin, ydv[i2]);
                        const float term = __fsub_rn(__fmul_rn(d, (float)dot), __fmul_rn(dm, mn[i2]));
                        acc[m][t][i2] = __fadd_rn(acc[m][t][i2], term);
                    }
                }
            }
        }
    };

    // Two register stages, one in flight while the other is multiplied; written out for an even and for an odd number
    // of stages (an odd run is one stage followed by an even run with the stages' roles swapped), so that no request
    // is ever made for a stage that does not exist.
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    constexpr std::false_type kMore{};
    constexpr std::true_type kLast{};
    const bool single = ODD && cnt == 1;  // wave-uniform
    issue(S0{}, 0, kMore);
    asm volatile("" ::: "memory");  // requests stay in stage order
    if (!single) {
        issue(S1{}, 1, kLast);
        asm volatile("" ::: "memory");
    }
    if constexpr (!GA) {
        // the LDS-direct copies are older than the tile requests: they have landed once at most those are outstanding
        if (single) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(NMAT * kTileLoads) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * NMAT * kTileLoads) : "memory");
        __builtin_amdgcn_s_barrier();  // no fence: a fence would wait for the outstanding weight tiles as well
        asm volatile("" ::: "memory");
    }
    if constexpr (ODD) {
        consume(S0{}, 0);
        if (!single) {
            issue(S0{}, 2, kLast);  // cnt >= 3
            asm volatile("" ::: "memory");
            int i = 1;
            auto two_stages = [&](auto last_c) {
                consume(S1{}, i);
                issue(S1{}, i + 2, kMore);
                asm volatile("" ::: "memory");
                consume(S0{}, i + 1);
                issue(S0{}, i + 3, last_c);
                asm volatile("" ::: "memory");
                i += 2;
            };
            while (i + (kUneven ? 4 : 2) < cnt) two_stages(kMore);
            if (kUneven && i + 2 < cnt) two_stages(kLast);
            consume(S1{}, i);
            if (last_exists) consume(S0{}, i + 1);
        }
    } else {
        // The next run of super-blocks replaces the one in LDS once every wavefront has multiplied its last stage of it
        // (the weight tiles of the next run's first two stages are already on their way: they do not depend on LDS).
        if constexpr (FLOW == 0) {
            // A single run, or runs of an even number of stages: run by run, the change of runs between two inner loops
            // (a conditional change inside the pipelined loop, as below, costs the Q6_K forms their registers: 256 and
            // spills against 120-130).  The last pair of stages of the launch is peeled off: no request past the end.
            const int runs = GA ? 1 : p.ranges;
            int i = 0;
            auto two_stages = [&](auto last_c) {
                consume(S0{}, i);
                issue(S0{}, i + 2, kMore);
                asm volatile("" ::: "memory");
                consume(S1{}, i + 1);
                issue(S1{}, i + 3, last_c);
                asm volatile("" ::: "memory");
                i += 2;
            };
            for (int rg = 0; rg < runs; ++rg) {
                if (rg > 0) {  // wave-uniform, the same in every wavefront
                    __syncthreads();
                    stage_range(rg);
                    b_range0 = rg * sb_per_range;
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's share of the copy (and its two stages of weight tiles)
                    __syncthreads();
                }
                const int i_stop = (rg + 1) * (cnt / runs) - (rg == runs - 1 ? (kUneven ? 4 : 2) : 0);
                while (i < i_stop) two_stages(kMore);
            }
            if (kUneven && i + 2 < cnt) two_stages(kLast);
            consume(S0{}, i);
            if (last_exists) consume(S1{}, i + 1);
        } else {
            // FLOW == 2: runs of an odd number of stages begin at either stage of a pair
            auto next_range = [&](int i) {
                if (GA || p.ranges == 1 || i == 0 || i % stages_per_range) return;  // wave-uniform, the same i in every wavefront
                __syncthreads();
                const int rg = i / stages_per_range;
                stage_range(rg);
                b_range0 = rg * sb_per_range;
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's share of the copy (and its two stages of weight tiles)
                __syncthreads();
            };
            int i = 0;
            for (; i + 2 < cnt; i += 2) {
                next_range(i);
                consume(S0{}, i);
                issue(S0{}, i + 2, kMore);
                asm volatile("" ::: "memory");
                next_range(i + 1);
                consume(S1{}, i + 1);
                issue(S1{}, i + 3, kMore);
                asm volatile("" ::: "memory");
            }
            next_range(i);
            consume(S0{}, i);
            next_range(i + 1);
            consume(S1{}, i + 1);
        }
    }

    // ---- the WPR wavefronts of a row tile meet in wave order; the first one stores ----
    if (WPR > 1) {
        if (kRedShares) __syncthreads();  // every wavefront has read its last activation tile
        if (h > 0) {
#pragma unroll
            for (int m = 0; m < NMAT; ++m)
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        red[(((((pair * (WPR - 1) + (h - 1)) * NMAT + m) * MT + t) * 4 + i) * 64) + lane] = acc[m][t][i];
        }
        __syncthreads();
    }
    if (h == 0 && !dead) {
        for (int wv = 1; wv < WPR; ++wv) {
#pragma unroll
            for (int m = 0; m < NMAT; ++m)
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc[m][t][i] = __fadd_rn(acc[m][t][i], red[(((((pair * (WPR - 1) + (wv - 1)) * NMAT + m) * MT + t) * 4 + i) * 64) + lane]);
        }
        const int64_t row = rt * 16 + r;
        if (row < p.rows) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int tok = 16 * t + 4 * kq + i;
                    if (tok < p.n) {
                        float v = acc[0][t][i];
                        if (NMAT == 2) v = silu_mul(v, acc[NMAT - 1][t][i], p.silu_mode);
                        p.y[(size_t)tok * (size_t)p.ldy + (size_t)row] = v;
                    }
                }
        }
    }
}

}  // namespace

namespace {

constexpr size_t kSkinnyLdsMax = 160 * 1024;

size_t skinny16_red_bytes(int nmat, int wpr, int mt) { return (size_t)(8 / wpr) * (wpr - 1) * nmat * mt * 4 * 64 * sizeof(float); }
// LDS of the form with the rows' tiles in LDS, `ranges` runs of super-blocks one after the other: with one tile of
// sixteen the partial sums lie behind the tiles, with more they share the tiles' bytes
size_t skinny16_lds_bytes(int nmat, int wpr, int64_t nb, int mt, int ranges) {
    const size_t tiles = (size_t)(nb / ranges) * mt * kPTileBytes, red = skinny16_red_bytes(nmat, wpr, mt);
    return mt > 1 ? (tiles > red ? tiles : red) : tiles + red;
}
// Runs of super-blocks the rows' tiles need to pass through LDS (1, 2 or 4; every wavefront must have a whole number
// of stages per run), or 0: they do not fit that way.
int skinny16_ranges(int nmat, int wpr, int64_t nb, int mt) {
    for (int ranges = 1; ranges <= 4; ranges *= 2) {
        if (ranges > 1 && (mt == 1 || nb % ((int64_t)wpr * ranges))) break;
        if (skinny16_lds_bytes(nmat, wpr, nb, mt, ranges) <= kSkinnyLdsMax) return ranges;
    }
    return 0;
}

template <int NMAT, int WPR, int FLOW, bool GA, int MT, int WT>
hipError_t launch_skinny16_one(const Skinny16Args& a, int ranges, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
    const int64_t rowtiles = (a.rows + 15) / 16;
    const size_t lds = GA ? skinny16_red_bytes(NMAT, WPR, MT) : skinny16_lds_bytes(NMAT, WPR, a.nb, MT, ranges);
    auto* kernel = &skinny16_kernel<NMAT, WPR, FLOW, GA, MT, WT>;
    static bool raised = false;  // per instantiation; the attribute belongs to the function, not to a launch
    if (!raised) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSkinnyLdsMax);
        if (e != hipSuccess) return e;
        raised = true;
    }
    Skinny16Args b = a;
    b.ranges = GA ? 1 : ranges;
    constexpr int RPW = 8 / WPR;
    const dim3 grid((unsigned)((rowtiles + RPW - 1) / RPW));
    if (start && stop) hipExtLaunchKernelGGL(kernel, grid, dim3(512), lds, stream, start, stop, 0, b);
    else MQ_LAUNCH(kernel, grid, dim3(512), lds, stream, b);
    return hipGetLastError();
}

// MT <= 2: the rows' tiles in LDS (in runs if need be), else from global memory a stage ahead; three and four tiles only
// from LDS (read a stage ahead they do not fit the registers).  Left out for their registers (256 and four to twelve
// spilled): pairs of four tiles with eight wavefronts per row tile, Q5_K and Q6_K pairs of two tiles read a stage ahead.  Not
// built although they would fit (106 to 240 registers, nothing spilled; not timed): Q6_K in runs of an odd number of stages and
// Q6_K pairs with one wavefront per row tile, which spilled while Q6_K multiplied by scale groups, and the Q5_K pair of four
// tiles in runs of an odd number of stages.
template <int NMAT, int WPR, int MT, int WT>
hipError_t launch_skinny16_form(const Skinny16Args& a, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
    const bool odd = (((a.nb + WPR - 1) / WPR) & 1) != 0;
    const int ranges = odd ? (skinny16_lds_bytes(NMAT, WPR, a.nb, MT, 1) <= kSkinnyLdsMax ? 1 : 0) : skinny16_ranges(NMAT, WPR, a.nb, MT);
    // (skinny16_applies knows the forms that are not built)
    if constexpr (WT == kWtQ6 && NMAT == 2 && WPR == 1) {
        return hipErrorInvalidValue;
    } else if constexpr (MT <= 2) {
        const bool ga = ranges != 1;  // (two tiles could also come in runs; read a stage ahead they cost no barrier)
        if constexpr (WT != kWtQ4 && NMAT == 2 && MT == 2) {  // two tiles of a Q5_K or Q6_K pair: not read a stage ahead
            if (ga) return hipErrorInvalidValue;
            if (odd) return launch_skinny16_one<NMAT, WPR, 1, false, MT, WT>(a, 1, stream, start, stop);
            return launch_skinny16_one<NMAT, WPR, 0, false, MT, WT>(a, 1, stream, start, stop);
        } else {
            if (odd) return ga ? launch_skinny16_one<NMAT, WPR, 1, true, MT, WT>(a, 1, stream, start, stop) : launch_skinny16_one<NMAT, WPR, 1, false, MT, WT>(a, 1, stream, start, stop);
            return ga ? launch_skinny16_one<NMAT, WPR, 0, true, MT, WT>(a, 1, stream, start, stop) : launch_skinny16_one<NMAT, WPR, 0, false, MT, WT>(a, 1, stream, start, stop);
        }
    } else if constexpr (WPR == 1 || (NMAT == 2 && MT == 4 && WPR == 8)) {
        return hipErrorInvalidValue;
    } else {
        if (ranges == 0) return hipErrorInvalidValue;
        if (odd) return launch_skinny16_one<NMAT, WPR, 1, false, MT, WT>(a, 1, stream, start, stop);  // (an odd stage count: one run only)
        if (((((a.nb + WPR - 1) / WPR) / ranges) & 1) == 0) return launch_skinny16_one<NMAT, WPR, 0, false, MT, WT>(a, ranges, stream, start, stop);
        if constexpr (WT == kWtQ6 || (WT == kWtQ5 && NMAT == 2 && MT == 4)) return hipErrorInvalidValue;  // (runs of an odd stage count)
        else return launch_skinny16_one<NMAT, WPR, 2, false, MT, WT>(a, ranges, stream, start, stop);
    }
}

template <int NMAT, int MT, int WT>
hipError_t launch_skinny16_wpr(const Skinny16Args& a, int wpr, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
    switch (wpr) {
        case 1: return launch_skinny16_form<NMAT, 1, MT, WT>(a, stream, start, stop);
        case 2: return launch_skinny16_form<NMAT, 2, MT, WT>(a, stream, start, stop);
        case 4: return launch_skinny16_form<NMAT, 4, MT, WT>(a, stream, start, stop);
        case 8: return launch_skinny16_form<NMAT, 8, MT, WT>(a, stream, start, stop);
    }
    return hipErrorInvalidValue;
}

template <int NMAT>
hipError_t launch_skinny16_tiles(const Skinny16Args& a, int wpr, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
    const int mt = (int)((a.n + 15) / 16);
    if (a.wtype == kTypeQ5K) {
        if (mt == 1) return launch_skinny16_wpr<NMAT, 1, kWtQ5>(a, wpr, stream, start, stop);
        if (mt == 2) return launch_skinny16_wpr<NMAT, 2, kWtQ5>(a, wpr, stream, start, stop);
        if (mt == 3) return launch_skinny16_wpr<NMAT, 3, kWtQ5>(a, wpr, stream, start, stop);
        if (mt == 4) return launch_skinny16_wpr<NMAT, 4, kWtQ5>(a, wpr, stream, start, stop);
        return hipErrorInvalidValue;
    }
    if (a.wtype == kTypeQ6K) {
        if (mt == 1) return launch_skinny16_wpr<NMAT, 1, kWtQ6>(a, wpr, stream, start, stop);
        if (mt == 2) return launch_skinny16_wpr<NMAT, 2, kWtQ6>(a, wpr, stream, start, stop);
        if (mt == 3) return launch_skinny16_wpr<NMAT, 3, kWtQ6>(a, wpr, stream, start, stop);
        if (mt == 4) return launch_skinny16_wpr<NMAT, 4, kWtQ6>(a, wpr, stream, start, stop);
        return hipErrorInvalidValue;
    }
    switch (mt) {
        case 1: return launch_skinny16_wpr<NMAT, 1, kWtQ4>(a, wpr, stream, start, stop);
        case 2: return launch_skinny16_wpr<NMAT, 2, kWtQ4>(a, wpr, stream, start, stop);
        case 3: return launch_skinny16_wpr<NMAT, 3, kWtQ4>(a, wpr, stream, start, stop);
        case 4: return launch_skinny16_wpr<NMAT, 4, kWtQ4>(a, wpr, stream, start, stop);
    }
    return hipErrorInvalidValue;
}

}  // namespace

// Whether a product of n rows (nine to 64) runs on skinny16_kernel: the wave split of the other decode kernels must be
// one of its own (a divisor of eight), and the form must be built
// (launch_skinny16_form returns an error for the others).
//   One and two tiles (up to 32 rows): always; the two tiles of a Q5_K or Q6_K gate/up pair only where they fit LDS in
//   one run; a Q6_K pair not with one wavefront per row tile.
//   Three and four tiles: not with one wavefront per row tile (more than 1,024 row tiles: the GEMM is faster from 33
//   rows -- 128256 x 4096 at 33 / 64 rows: 93 / 108 us against 102 / 126); the tiles must pass through LDS in at most four
//   runs of whole stages (in one run where a wavefront's stage count is odd or the split uneven); a pair of four tiles not with eight
//   wavefronts per row tile; in runs of an odd number of stages no Q6_K form and no Q5_K pair of four tiles.
bool skinny16_applies(int64_t nb, int64_t rowtiles, bool swiglu, int64_t n, int wtype) {
    const int wpr = dense_lds_wpr(nb, rowtiles);
    if (!wpr || n < 1 || n > 64 || (wtype != kTypeQ4K && wtype != kTypeQ5K && wtype != kTypeQ6K)) return false;
    const int nmat = swiglu ? 2 : 1, mt = (int)((n + 15) / 16);
    if (wtype == kTypeQ6K && swiglu && wpr == 1) return false;
    if (nb % wpr && !skinny16_uneven(nmat, wpr, skinny16_lds_bytes(nmat, wpr, nb, mt, 1) > kSkinnyLdsMax, mt)) return false;
    if (mt <= 2) return !(wtype != kTypeQ4K && swiglu && mt == 2) || skinny16_lds_bytes(2, wpr, nb, 2, 1) <= kSkinnyLdsMax;
    if (wpr == 1 || (swiglu && mt == 4 && wpr == 8)) return false;
    if (nb % wpr || ((nb / wpr) & 1)) return skinny16_lds_bytes(nmat, wpr, nb, mt, 1) <= kSkinnyLdsMax;  // an uneven split, an odd stage count: the tiles in one run
    const int ranges = skinny16_ranges(nmat, wpr, nb, mt);
    if (!ranges) return false;
    const bool odd_runs = (((nb / wpr) / ranges) & 1) != 0;
    return !odd_runs || !(wtype == kTypeQ6K || (wtype == kTypeQ5K && swiglu && mt == 4));
}

bool skinny16_one_run(int64_t nb, int64_t rowtiles, bool swiglu, int64_t n) {
    const int wpr = dense_lds_wpr(nb, rowtiles);
    return wpr && skinny16_lds_bytes(swiglu ? 2 : 1, wpr, nb, (int)((n + 15) / 16), 1) <= kSkinnyLdsMax;
}

hipError_t launch_skinny16(const Skinny16Args& a, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
    if (a.rows <= 0 || a.nb <= 0 || a.n < 1 || a.n > 64 || !a.y || !a.w0 || !a.ap) return hipErrorInvalidValue;
    const int64_t rowtiles = (a.rows + 15) / 16;
    if (!skinny16_applies(a.nb, rowtiles, a.w1 != nullptr, a.n, a.wtype)) return hipErrorInvalidValue;
    const int wpr = dense_lds_wpr(a.nb, rowtiles);
    if (a.w1) return launch_skinny16_tiles<2>(a, wpr, stream, start, stop);
    return launch_skinny16_tiles<1>(a, wpr, stream, start, stop);
}

}  // namespace mq
