/*
 * mi355_q4k_debug.h -- verification hooks and measurement instruments of libmi355q4k.so.
 *
 * Exported by the same library as the entry points of mi355_q4k.h, kept apart from them: a DenseCore host binds
 * mi355_q4k.h; tests and benchmarks also include this file.  None of these calls changes what a product entry point
 * computes; mq_debug_set_dense_lds selects between kernels that return the same bits up to 16 rows and agree to rounding beyond.
 */
#ifndef MI355_Q4K_DEBUG_H
#define MI355_Q4K_DEBUG_H

#include "mi355_q4k.h"

#ifdef __cplusplus
extern "C" {
#endif

/* ---- verification hook -------------------------------------------------------------
 * Runs the production matmul kernel with its per-super-block integer sums
 * written out: dot_scaled_dev / min_dot_dev int32 [rows][n][cols/256], the two
 * integers every reference kernel forms before touching floating point
 * (core/src/llm/matmul/kquant_batched_kernels.h:285-297).  Mirrors the
 * reference's ...ForTest hooks (core/src/llm/moe/native.cpp:5107-5636). */
int mq_debug_block_sums(const mq_weight* w, const float* x_dev, int64_t n, int64_t ldx, int32_t* dot_scaled_dev,
                        int32_t* min_dot_dev, float* y_dev, int64_t ldy, void* stream);

/* The expert-grouped work list ("gather tokens by expert") that the grouped kernels read, written out entry by
 * entry: triples_dev int32 [n * top_k][3] = (expert, token, k) in list order, count_dev int32 [1] = entries (pairs
 * whose id is outside [0, n_experts) are dropped).  The reference's list is sorted by (expert, token, k)
 * (Qwen35BuildMoEAssignments, core/src/llm/moe/native.cpp:1664-1733).  Pass ids_dev int32 [n][top_k] to group given
 * ids (the grouping launch of mq_mul_mat_id_q4k and of the two expert nodes on the decode launches) or logits_dev fp32 [n][n_experts] to
 * route and group in the one launch mq_moe_layer_q4k uses above eight tokens; the other pointer NULL. */
int mq_debug_moe_groups(const float* logits_dev, const int32_t* ids_dev, int64_t n_experts, int64_t n, int top_k,
                        int32_t* triples_dev, int32_t* count_dev, void* stream);

/* The plan of the expert-grouped GEMM as its launch (or, beyond 512 experts or 65,536 pairs, its two launches) lays it out for the given
 * ids, with every token of a shared expert as one more group if asked for: plan_dev int32 [layout_out[2]], and the work list it leaves for
 * a down stack that the GEMM does not take, as mq_debug_moe_groups writes it.  plan[0] items, [1] tiles of sixteen rows, [2] those of routed
 * pairs, [4 + 3 i ..] expert (-1: the shared one), first tile and tiles of item i; from layout_out[0] on the token of each of the tiles' rows,
 * from layout_out[1] on its output row token * slots + slot, -1 for padding.  plan_dev NULL: the layout alone. */
int mq_debug_moe_plan(const int32_t* ids_dev, int64_t n_experts, int64_t n, int top_k, int shared, int item_tiles, int32_t* triples_dev,
                      int32_t* count_dev, int32_t* plan_dev, int64_t* layout_out, void* stream);

/* The fp32 intermediate the last mq_moe_layer_q4k / mq_ffn_swiglu_q4k call on this stream left in the library's
 * workspace, copied out: for the MoE layer the hidden rows silu(gate . x) * (up . x) as [n][top_k (+1 with a shared
 * expert)][inter], for the dense FFN [n][inter].  `count` floats, no more than that call left (MQ_ERR_INVALID).
 * MQ_ERR_STATE where the rows are not there: no such call yet, a later product used the workspace, or the layer took the
 * expert-grouped GEMM, which forms them in its tiles' order.  Replays of a captured call do not count as calls.  A ...ForTest hook like
 * mq_debug_block_sums. */
int mq_debug_moe_hidden(float* hidden_out_dev, size_t count, void* stream);
/* Device addresses of a decoder handle's exchange buffers after a step (the LAST layer's values): qkv [n][qkv_rows],
 * o [n][hidden], logits [n][n_experts], hidden rows [n][top_k (+1)][inter], MoE output y [n][hidden].  Any may be NULL. */
int mq_debug_decoder_buffers(mq_decoder* d, float** qkv_dev, float** o_dev, float** logits_dev, float** hidden_dev,
                             float** y_dev);

/* ---- launch census -------------------------------------------------------------------
 * When enabled, every matmul-kernel launch carries a start/stop HIP event pair that receives the
 * dispatch's own begin and end timestamps; mq_census_read synchronises and returns the kernel durations.  The GPU
 * counterpart of the reference's matmul dispatch census of (path, shape, wall ns)
 * (core/src/llm/matmul/gemv_exec.cpp:203-276).  Off by default. */
#define MQ_KIND_DENSE 0          /* one dense matrix                     */
#define MQ_KIND_DENSE_SWIGLU 1   /* gate + up fused, dense               */
#define MQ_KIND_GROUPED 2        /* expert-routed                        */
#define MQ_KIND_GROUPED_SWIGLU 3 /* expert-routed gate + up fused        */
#define MQ_KIND_COUNT 4
int mq_census_enable(int on);
int mq_census_reset(void);
int mq_census_read(int kind, double* avg_us, double* min_us, double* max_us, int64_t* count);

/* Debug switch: dense products of up to 16 rows normally run on the kernel that stages the quantized activations
 * in LDS once per workgroup (and, for up to four fp32 rows, quantizes them itself), and expert-grouped launches
 * with many groups on the kernel that gathers a group's rows into LDS once per eight wavefronts; on = 0 keeps
 * both on the kernel that reads its operand from global memory at every stage, on = 5 only the expert-grouped
 * ones; bit 3 (on = 9) makes gate and up at prefill widths two GEMM launches and a SwiGLU pass instead of the
 * one launch that stores silu(gate) * up; bits 8..11 force the activation tiles per item of the expert-grouped GEMM (2,
 * 4 or 8; 0 = chosen by the rows per expert); bit 12 keeps dense products of nine to 64 rows on the kernels
 * that multiply them as token tiles of eight (or on the GEMM) instead of the one that takes them as tiles of sixteen.  They
 * return the same bits (tests/test_gpu_dense_lds.py, tests/test_gpu_grouped_lds.py, tests/test_gpu_prefill.py), except that bits 0 and 12
 * also turn off the choice by estimate between 17 and 64 rows, and bit 3 lets K be cut into runs: a product that so changes between
 * the decode kernels and the GEMM, or its GEMM's shape, agrees to rounding.  Returns the previous setting of bit 0.  No counterpart in the reference. */
int mq_debug_set_dense_lds(int on);

/* Launch shape that the matrix-core GEMM takes for a product of n rows (pair 1: for gate and up in one launch, 2: ahead of a down product), for a 256-unit
 * device before mq_init.  shape_out: 64-row workgroups (1) or 128-row ones (0), runs of K, super-blocks per run, activation tiles per
 * workgroup, workgroup rows, workgroup columns, whether the one launch is taken (1 where pair == 0), the estimate in ns.  Planes of
 * partial sums have rows of four floats, so for a row count that does not divide by four this is the best shape without runs; a product of
 * such a matrix is launched in the shape of the row count padded to four where that one's estimate is less. */
int mq_debug_gemm_shape(int wtype, int64_t rows, int64_t cols, int64_t n, int pair, int* shape_out);

/* The first six of these for the launch that a GEMM product by itself makes, padded rows and Q8_0 weights included. */
int mq_debug_gemm_launch(int wtype, int64_t rows, int64_t cols, int64_t n, int* shape_out);

/* Kernels that a dense product of n rows (pair 1: gate and up in one call; 2: the down product of an FFN whose gate and up run on the
 * GEMM) runs on, for a 256-unit device before mq_init.  path_out:
 * 0 passes of eight or sixteen rows, 1 tiles of sixteen, 2 the matrix-core GEMM; wavefronts per row tile of the passes, and of the
 * tiles of sixteen (0: not built for this product).  Q8_0 (pair == 0): 0 or 2; wavefronts per row tile of the passes; activation tiles
 * per workgroup of the GEMM. */
int mq_debug_dense_path(int wtype, int64_t rows, int64_t cols, int64_t n, int pair, int* path_out);

/* Whether the expert products of a MoE block run on the expert-grouped GEMM (1) or on the decode launches (0), for a 256-unit device before
 * mq_init.  path_out: gate/up and down of mq_moe_layer_q4k, then mq_moe_gateup_swiglu_q4k and mq_moe_down_weighted_q4k on such stacks. */
int mq_debug_moe_path(int gate_type, int down_type, int64_t n_experts, int64_t hidden, int64_t inter, int64_t n, int top_k, int* path_out);

/* Measurement instrument: while on != 0 every compute and routing launch of the library is replaced by a kernel with
 * an empty body and the same grid, block and LDS size (weight set-up and launches that carry timing events are
 * not).  A graph captured in this state has the launches of the real one and none of their work: its replay time
 * is what the launches alone cost.  Outputs are not written while it is on.  Returns the previous setting.  No
 * counterpart in the reference. */
int mq_debug_set_skeleton(int on);

#ifdef __cplusplus
}
#endif
#endif
