/*
 * sgemm_debug.h - profiling aids of libsgemm.so.  Not part of the drop-in interface of sgemm.h: nothing here has a
 * counterpart in the reference, and a caller of the library never needs it.  bench.py uses both to produce the
 * time-stamp tables and the read-only ceiling under profiles/.
 */
#ifndef SGEMM_DEBUG_H
#define SGEMM_DEBUG_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Profiling aid, no counterpart in the reference.  While a buffer is set, every launch of the LDS-ring GEMM
 * kernels (per-tile and persistent), of the mid-batch (whole lines or not) and wide-tile GEMM kernels and of the 2:4
 * kernels takes the next grid * 8 words of it and each workgroup leaves eight 64-bit
 * words there when it is done: [0] kernel entry, [1] prologue DMAs issued, [2] first stage landed, [3] last stage
 * consumed, [4] outputs stored and acknowledged - 10 ns ticks of the device's constant 100 MHz clock -
 * [5], [6] shader clock at entry and end, [7] XCC_ID << 32 | HW_ID.  Launches that no longer fit leave nothing.
 * A launch recorded into a HIP graph keeps its slice on every replay.  Process-wide; set it from one thread while
 * no other thread launches.  sg_debug_stamps(NULL, 0) switches the stamps off again. */
int sg_debug_stamps(unsigned long long* device_buffer, size_t n_words);

/* The GEMM of sg_skinny_gemm_rowcol on the wide-tile kernel with a given tile, for tests and timings of single tiles: the
 * library chooses between them by itself above 128 rows.  The tile is 32 * row_tiles weight rows (row_tiles 4..8) by
 * 32 * m_blocks activation rows (8, or 4 with row_tiles 4 and 8); split_k > 1 sums its partials in a second launch.
 * scale, row_scales and col_scales may be NULL; k a multiple of 16 beyond 128. */
int sg_debug_wide_gemm(const uint8_t* A, const uint8_t* B, void* D_bf16, const float* scale, const float* row_scales,
                       const float* col_scales, int m, int n, int k, int b_stride, int row_tiles, int m_blocks, int split_k,
                       void* stream);

/* Which wide tile sg_skinny_gemm_auto - with factors: sg_skinny_gemm_rowcol with row or column factors - launches for the
 * shape and row stride: out = {row_tiles, m_blocks, split_k} as sg_debug_wide_gemm takes them, or three zeros where it
 * launches something else. */
int sg_debug_wide_choice(int m, int n, int k, int b_stride, int factors, int out[3]);

/* The GEMM of sg_debug_wide_gemm on the kernel for rows that start off their 128-byte lines: the tile is
 * 8 * waves * row_tiles weight rows by 32 * m_blocks activation rows, (waves, row_tiles, m_blocks) one of (4, 2, 2),
 * (8, 2, 2), (8, 2, 4), (8, 2, 6) and (8, 3, 4); a K split sums its partials in a second launch.  Any k and stride the
 * library takes, also on whole lines. */
int sg_debug_line_gemm(const uint8_t* A, const uint8_t* B, void* D_bf16, const float* scale, const float* row_scales,
                       const float* col_scales, int m, int n, int k, int b_stride, int waves, int row_tiles, int m_blocks,
                       int split_k, void* stream);

/* ... and which tile of that kernel sg_skinny_gemm_auto - with factors: sg_skinny_gemm_rowcol - launches for the shape and
 * row stride: out = {waves, row_tiles, m_blocks, split_k}, or four zeros where it launches something else. */
int sg_debug_line_choice(int m, int n, int k, int b_stride, int factors, int out[4]);

/* The GEMM of sg_skinny_gemm_rowcol at up to 32 rows on one of the skinny kernels for rows that start off their 128-byte
 * lines, k beyond 256.  resident = 0: a workgroup of `waves` waves per tile of 16 * row_tiles weight rows, K shared among them
 * and among split_k workgroups, `depth` ring slots a wave: (row_tiles, depth) = (1, 4), (2, 3) and (2, 4), (4, 3) - from 9 rows on;
 * above 16 rows (1, 4), (2, 4) and (4, 3).  resident = 1: one workgroup per CU with all activations in LDS, whose waves own
 * whole 16-row tiles (row_tiles and split_k 1, depth 3 or 4). */
int sg_debug_skinny_line_gemm(const uint8_t* A, const uint8_t* B, void* D_bf16, const float* scale, const float* row_scales,
                              const float* col_scales, int m, int n, int k, int b_stride, int resident, int waves, int row_tiles,
                              int depth, int split_k, void* stream);

/* ... and what sg_skinny_gemm_auto launches of them for the shape and row stride: out = {waves, row_tiles, depth, split_k,
 * resident}, or five zeros where it launches something else. */
int sg_debug_skinny_line_choice(int m, int n, int k, int b_stride, int out[5]);

/* Profiling aid, no counterpart in the reference: reads the n x k weight matrix B (row stride b_stride, k % 1024 == 0)
 * the way the persistent LDS-ring GEMM streams it - one workgroup per CU walking row tiles, eight waves sharing K,
 * direct-to-LDS loads with the streaming hint, two 4 KB slots per wave - and does nothing with it.  Its duration is the
 * ceiling of that access pattern on the device: what a GEMM's streaming phase is measured against.  segment_bytes is
 * what one load instruction takes contiguously from one row: 256 (4 rows per instruction - the GEMM's own pattern),
 * 512 (2 rows) or 1024 (1 row). */
int sg_debug_read_stream(const uint8_t* B, int n, int k, int b_stride, int segment_bytes, void* stream);

/* Profiling aid, no counterpart in the reference: what a CU takes in through direct-to-LDS loads when part of its
 * stream misses the XCD's L2 and part of it hits.  `workgroups` workgroups of `waves` waves (1, 2, 4, 8 or 16) issue
 * 1 KB loads (8 rows x 128 B, rows 8 KB apart - the mid-batch GEMM's pattern) with `depth` (4, 8 or 16, at most
 * 128 / waves) instructions in flight per wave for `ticks` x 10 ns and count them: counts[0] += loads of the cold
 * stream (a region of its own per wave out of `cold`, streaming hint), counts[1] += loads of the hot stream (one window
 * per XCD out of `hot`, walked by all its workgroups; make hot_bytes / 8 fit an L2).  cold_waves >= 0: waves below it
 * stream cold, the others hot; cold_waves < 0: every wave alternates hot_per_cold hot loads with one cold one.
 * The caller zeroes counts (two 64-bit words in device memory) and reads them after the stream has finished. */
int sg_debug_cu_ingest(const uint8_t* cold, size_t cold_bytes, const uint8_t* hot, size_t hot_bytes, int workgroups, int waves,
                       int cold_waves, int hot_per_cold, int depth, int ticks, unsigned long long* counts, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* SGEMM_DEBUG_H */
