/*
 * w4a8_probe.h -- measurement probes exported by libw4a8_mi355x.so, not part of the W4A8 path.
 *
 * No counterpart in the reference. bench.py --read-floor uses it to time one launch of a plain
 * streaming-read kernel over B bytes (the floor a decode GEMV call of B weight bytes is read
 * against). Conventions as in w4a8_mi355x.h: device pointers, a hipStream_t as void*, 0 on success.
 */
#ifndef W4A8_PROBE_H
#define W4A8_PROBE_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Read `bytes` (a multiple of 16, under 4 GiB) of buf with 16-byte non-temporal loads,
 * loads_per_thread (1, 4, 8 or 16) per thread and pass, workgroups of `threads` (64, 256, 512 or
 * 1024). grid = 0: a one-shot grid covering the buffer once; grid > 0: that many workgroups striding
 * over it. sink: 4 device bytes a never-taken store may write (it keeps the loads alive). Returns 1
 * on bad arguments, 3 on a launch error. */
int w4a8_probe_read(const void* buf, int64_t bytes, int loads_per_thread, int threads, int grid, uint32_t* sink,
                    void* stream);

/* The tile (rows << 16 | columns) that a dense prefill call of w4a8_linear or w4a8_gemm runs on, given its
 * activations in the GEMM's operand order or not; 0 for M = 0 and for NVFP4 (whose kernel has tiles of its
 * own); minus the status code on bad arguments. Host-only. For tests that mean to run a certain tile. */
int w4a8_probe_prefill_tile(int64_t M, int64_t N, int64_t K, int scale_fmt, int has_zeros, int wfmt,
                            int64_t group_size, int silu, int operand_order);

#ifdef __cplusplus
}
#endif

#endif
