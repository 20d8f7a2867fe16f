/* Where the fp32 GEMM's tile loads (gemm_x3.hip) read: runs of four floats, in
 * bytes from the tile's first element.  Plain arithmetic, host and device, so that
 * a test can go through all of it on the CPU.
 *
 * CONTIG tiles have k along a row (rows of A, or of a transposed B), the others
 * have a row per k.  Rows past the matrix repeat its last one, runs past its last
 * column start at the first (both feed outputs that are not stored).  So no run
 * leaves the matrix while its columns (K in CONTIG tiles) are a multiple of 4, and
 * else the last one does by at most 12 bytes. */
#ifndef TM_X3_RUNS_H
#define TM_X3_RUNS_H

#include <stdint.h>

#ifdef __HIP__
#define TM_RUN __host__ __device__ __forceinline__
#else
#define TM_RUN inline
#endif

/* The run at (row, col) of a tile with `left` rows (CONTIG) or columns of the
 * matrix from its first element on */
template <bool CONTIG>
TM_RUN uint32_t x3_run(int64_t ld, int row, int col, int left) {
  return 4 * (CONTIG ? (uint32_t)((row < left ? row : left - 1) * ld) + col
                     : (uint32_t)(row * ld) + (col < left ? col : 0));
}
/* and in the last k-step, with `k_left` of its k inside the matrix: runs and rows
 * past them read the first (the caller replaces them by zeros) */
template <bool CONTIG>
TM_RUN uint32_t x3_last_run(uint32_t run, int64_t ld, int row, int col, int k_left) {
  if (CONTIG) return col < k_left ? run : run - 4 * col;
  return row < k_left ? run : run - 4 * (uint32_t)(row * ld);
}

#endif
