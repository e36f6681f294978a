/* Measurement aids of libdgpp_amd.so: A/B switches and streaming probes used by the benchmark and by the tests that
 * compare kernel forms. Nothing here is part of the drop-in launcher surface (dgpp_amd.h does not include this
 * file) and no product caller needs it. */
#ifndef DGPP_AMD_BENCH_H
#define DGPP_AMD_BENCH_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Bench A/B switches, process-wide relaxed atomics (a set that races a launch is defined: the launch takes the old or
 * the new value), 0 everywhere = the product behaviour. They are inert unless the process opted in through the
 * environment (DGPP_AMD_BENCH=1, see dgpp_tune_enabled); a library built with -DDGPP_NO_TUNE leaves them out
 * (dgpp_tune_set stores nothing, dgpp_tune_get returns 0). The reference keeps such a switch in its launcher header
 * too: moe_set_fp8_ldm, src/kernels/glm_moe_launch.hpp:90. key 0: preferred chunks per lane of the row geometry (0 =
 * default 4); key 1: slots of one expert a decode-slot block serves together (0 = default: 2 gate/up, 4 down; 1 = one
 * slot per block); key 2: row steps per block of the slot launches (0 = automatic); key 3: 1 stages activations before
 * any weight load is issued (default: activation loads, first weight pass, LDS commit); key 4: 1 keeps the layer
 * driver on the two-launch down + accumulate form; key 5: 2 moves every GEMV launcher to the matrix-core form, 1 keeps
 * the dense launchers on the vector core at every row count (default: the dense launchers choose by rows, matrix size
 * and workspace); key 6: 1 makes the layer driver compute the slot order for small decode batches too (default:
 * batches of at most 128 routed slots find the sharers of an expert by ballot, no order); key 7: 1 keeps the selection
 * of a one-token step a launch of its own (default: repeated in the gate/up blocks,
 * dgpp_launch_moe_select_gate_up_swiglu); key 8: row tiles an XCD takes for one token before it turns to the next
 * token in the token-major down + accumulate launch (0 = automatic: 1 from 64 routed slots on, else plain token-major
 * order); key 9: a block-FP8 shared expert's passes of the layer driver. 0 = the routed experts' launches take them where
 * dgpp_bench_merged_passes says so; elsewhere, and with any other value but 5 and 6, launches of their own: 1 on the caller's
 * stream, 2 on a second stream beside the routed passes at every batch size (default: from three tokens on in a captured step
 * or with more than 32 M shared weights, else from sixteen on); 3 and 4 keep one stream and never / always fold the
 * accumulation into the shared down pass (default: at one token); 5 and 6 merge gate + up or both passes wherever they have that form; key 10: 2 or 4 runs the router's token-tiled score
 * kernel at every batch size with that many tokens per wavefront, 16 or 32 the one on the matrix core with tiles of
 * that many (0 = automatic: tiled from 32 rows on, 4 tokens from 128 rows on, the matrix core where its blocks' walk
 * is shorter than the sums in lanes); key 11: the form of the dense matrix-core launch below the tiles: 4 streamed
 * wherever the rows are whole 16-byte vectors, 1 to 3 not streamed; without a workspace 1 row tiles, 2 the four parts
 * of K side by side inside a block of four row groups, 3 of two for up to eight rows (0 = automatic: streamed except
 * where another form fills the chip better; else four row groups while the row tiles fit one round of the chip, two up
 * to a round and a quarter); key 12: 1 makes dgpp_launch_moe_slot_chain* run the launches the one-launch chain stands
 * for, 2 makes the layer driver take the one-launch chain for small routed-only decode batches (default: the driver
 * runs the launches; the chain measured slower); key 13: row steps per wavefront of the chain's down part (0 =
 * automatic); key 14: the fused gate + up matrix-core grouped launch: 1 = every wavefront walks both matrices in turn,
 * 2 = the block's wavefronts split into gate walkers and up walkers (0 = automatic: split while the grid is at most
 * 2048 blocks); key 15: the forms for many activation rows. The dense and grouped matrix-core launches: 1 = the 16-row
 * form, 2 = tiles of 128 activation rows wherever the rows are 16-byte aligned, 3 = grouped passes of 32 there, 5
 * and 6 = dense tiles of 64 and of 32 (0 = automatic: dgpp_bench_dense_tile_rows, dgpp_bench_grouped_takes_narrow,
 * dgpp_bench_grouped_takes_tiles). The MXFP8 GEMM: 1 = the 16-row form, 2 - 4 = tiles of 32 x 64, 64 x 64 or 64 x 128 (weight x activation rows) through registers,
 * 5 - 9 = of 32 x 64, 64 x 64, 64 x 128, 128 x 64 or 128 x 128 through a ring of LDS stages (0 = automatic: dgpp_bench_mxfp8_form);
 * key 16: blocks that share the passes of a segment and a row tile in the grouped tiles (0 = automatic); key 17: the
 * MXFP8 shared expert's projections of more than 64 rows on the layer driver's second stream: 1 = the form that is
 * faster alone, 2 = the tiles (0 = automatic). Outputs do not depend on keys 1 - 4 and 6 - 17; keys 0 and 5 change the
 * fp32 summation order (every GEMV launcher follows them alike, so the launchers stay bitwise twins of each other). */
void dgpp_tune_set(int key, int value);
int dgpp_tune_get(int key);
/* 1 when the process opted in: the switches take values only if the environment held DGPP_AMD_BENCH=1 at the first
 * call of dgpp_tune_set / dgpp_tune_enabled (read once). Without it dgpp_tune_set stores nothing and every launcher
 * runs its measured default, whatever any component of the process calls. */
int dgpp_tune_enabled(void);

/* How many launches took a form of key 15's tiles so far, counted in a process that enabled the switches. */
int dgpp_bench_tiled_launches(void);
/* Likewise by form: 0 those, 1 the grouped passes of 32 rows, 2 streamed dense products, 3 dense products whose parts of K were
 * split over a workspace, 4 passes of the layer driver that took the routed and the shared expert in one launch. */
int dgpp_bench_form_launches(int form);

/* Activation rows to a tile, 128, 64 or 32, of the form that a dense matrix-core launch of m rows takes by its default rule (16-byte
 * aligned rows), or 0: a form of 16-row passes (streamed; or with its K parts in one block or split over a workspace). fmt: 0 block
 * FP8, 1 MXFP8, 2 NVFP4, 3 MXFP4; act_nvfp4: NVFP4 activations; beside: another product runs beside it; workspace: the caller's holds
 * the parts of K. Host arithmetic only. */
int dgpp_bench_dense_tile_rows(int fmt, int act_nvfp4, int m, int n, int k, int beside, int workspace);
/* The line, 1 above it, from which on the 128-row tiles take a launch of NVFP4 activations, no launch splits its K parts over a workspace, and a
 * plain launch does not stream. */
int dgpp_bench_dense_takes_tiles(int fmt, int m, int n, int k);
/* Likewise for a grouped matrix-core launch, where dgpp_bench_grouped_takes_narrow does not say 1: over n_segs
 * segments (act_nvfp4: NVFP4 activations; gate_up: gate and up in one launch) of max_rows rows at most and total_rows
 * together (0: the caller does not know), of which the last long_segs have max_rows: 1 = tiles of up to 128 activation
 * rows, 0 = the 16-row form. */
int dgpp_bench_grouped_takes_tiles(int fmt, int act_nvfp4, int gate_up, int n_segs, int k, int max_rows, int total_rows,
                                   int long_segs);
/* Whether that launch, of n weight rows, takes the passes of 32 rows: only if total_rows is known. */
int dgpp_bench_grouped_takes_narrow(int fmt, int act_nvfp4, int gate_up, int n_segs, int n, int k, int max_rows, int total_rows,
                                    int long_segs);
/* Which form the MXFP8 GEMM takes: 0 the 16-row one, 1 to 8 the tiles that key 15 numbers from 2 on; -1: k out of range. */
int dgpp_bench_mxfp8_form(int m, int n, int k);
/* How many passes of a decode step of the layer driver take the routed and a block-FP8 shared expert in one launch: 2 gate + up and
 * down with the accumulation, 1 gate + up, 0 neither. fmt: 0 block FP8, 2 NVFP4, 3 MXFP4; captured: on a stream that is being captured;
 * down_fits: the row widths have that form of down. Host arithmetic only. */
int dgpp_bench_merged_passes(int fmt, int tokens, int top_k, int n_experts, int hidden, int inter, int shared_inter, int captured,
                             int down_fits);
/* What a block of the grouped launch's 128-row form works on (the last long_segs of the table's segments are known to
 * have max_rows rows): place[0 .. 3] = segment (-1: nothing), row tile, first pass and step of its passes of 128 rows.
 * Returns the number of blocks; block b runs on XCD b % 8. Host arithmetic only. */
int dgpp_bench_tiled_place(int n_segs, int long_segs, int row_tiles, int max_rows, int block, int32_t* place);

/* How many items the passes of a grouped launch of known rows are sorted into (0: dealt by segment): no fewer than a
 * table of total_rows rows has passes of `cols` (128 or 32) rows. blocks: of that launch. -1: arguments out of range.
 * Host arithmetic only. */
int dgpp_bench_tiled_plan(int n_segs, int long_segs, int row_tiles, int max_rows, int64_t total_rows, int cols, int64_t* blocks);

/* Measurement aid with no counterpart in the reference: a plain streaming copy of `bytes`
 * (a multiple of 16; both pointers 16-byte aligned) on `stream`. A profiler's HBM byte counters
 * are calibrated against it: it reads `bytes` and writes `bytes`, nothing else. */
int dgpp_probe_copy(void* dst, const void* src, size_t bytes, void* stream);

/* A plain streaming READ of `bytes` (a multiple of 16, 16-byte aligned) on `stream`: 16-byte loads, eight in flight
 * per lane, nothing stored (`sink`, at least 8192 words, is written only for a checksum no input produces). `blocks`
 * blocks of 256 threads (0 = 2048, at most 8192); span != 0 gives every block one contiguous span of the buffer, span == 0
 * lets the whole grid stride through it together. The rate it reaches is the ceiling of a weight stream on this chip;
 * nontemporal != 0 uses the nontemporal load form the GEMV kernels use where a launch reads its weights once. */
int dgpp_probe_read(const void* src, size_t bytes, void* sink, int nontemporal, int blocks, int span, void* stream);

#ifdef __cplusplus
}
#endif
#endif
