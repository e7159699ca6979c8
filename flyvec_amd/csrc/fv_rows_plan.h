/* When the dense launch of a training step visits only the rows of the matrix somebody needs (fv_train_rows.h): the part
 * of the rule that looks at sizes, and how the demand for clear launches grows. Plain C; the CPU tests evaluate it. */
#pragma once

#include <stdint.h>

/* Where visiting rows pays, by the bytes of the matrix and the window positions of a minibatch per row of it. Measured:
 * time per step of the launch over every row / that of the rows form, Zipf tokens (1.05), K = 72, 128, 300, 600 (V up to
 * 60000; "-": no such size):
 *   MiB  0.15 positions        0.6                   1.5                   4                     8
 *   3    1.08 1.03 -    -      1.07 1.03 1.05 1.05   1.07 1.03 1.05 1.06   1.04 1.01 1.05 1.06   1.03 1.00 1.05 1.04
 *   6    1.09 1.11 1.07 -      1.09 1.03 1.08 1.04   1.05 1.04 1.06 1.05   1.04 1.00 1.01 1.04   1.02 1.00 1.01 1.01
 *   8    1.09 1.09 1.06 -      1.09 1.07 1.06 1.06   1.02 1.04 1.05 1.05   0.99 0.99 1.02 1.02   1.02 0.98 1.02 1.03
 *   12   1.09 1.10 1.10 1.08   1.06 1.07 1.06 1.05   1.01 1.02 1.02 1.02   0.99 1.00 1.00 1.00   0.99 1.00 1.01 1.01
 *   16   1.08 1.09 1.07 1.08   1.00 1.04 1.02 1.04   0.96 0.97 0.97 0.99   0.97 0.97 0.98 0.97   -    1.00 1.02 1.01
 *   20   1.02 1.07 1.09 1.09   0.94 1.02 1.02 1.02   0.98 0.96 0.96 0.98   0.96 1.00 1.02 1.00   -    1.00 1.00 1.02
 *   24   1.04 1.06 1.10 1.09   0.93 0.98 1.00 1.03   0.96 0.97 0.97 0.99   0.97 1.01 1.03 1.04   -    -    1.02 1.04
 *   28   1.02 1.03 1.12 1.11   0.94 0.96 1.03 1.03   0.98 1.02 1.02 1.02   -    1.00 1.06 1.05   -    -    1.02 1.04
 *   40   -    1.12 1.26 1.29   -    1.02 1.16 1.14   -    1.04 1.15 1.15   -    1.01 1.08 1.11   -    -    1.05 1.06
 * and 64 MiB 1.10 to 1.6 (K = 200, 400, 1000; 1.03 at 20 positions), 400 MB 1.10. Beside Zipf tokens uniform ones, which
 * touch more rows: as a rule 0.02 to 0.05 less. At 22 positions 3 to 8 MiB give 0.93 to 1.02, 28 and more 1.01 to 1.03.
 * The valley from 14 to 26 MiB: so much fits the eight L2s (4 MB each) where a row is always updated by the same block,
 * and less where any block visits it (what the times suggest; not counted). With 8 positions a row nearly every row is
 * visited anyway. Below 4 MiB a step gains 1 to 2 us at most, and loses as much at 20 positions. */
#define FV_ROWS_LEAST_BYTES (4ull << 20)
#define FV_ROWS_LEAST_LDK 32u /* (the lists take 16 bytes per row: an eighth of a matrix this narrow) */
#define FV_ROWS_NARROW_LDK 100u

static inline int fv_rows_pay(uint64_t n_rows, uint32_t ldk, uint64_t positions) {
  const uint64_t bytes = n_rows * ldk * 4, mib = 1ull << 20;
  const int narrow = ldk < FV_ROWS_NARROW_LDK;
  if (ldk < FV_ROWS_LEAST_LDK || bytes < FV_ROWS_LEAST_BYTES) return 0;
  if (bytes < 9 * mib) return positions <= 8 * n_rows;
  if (bytes < 14 * mib) return positions <= 2 * n_rows;
  if (bytes < (narrow ? 40 : 26) * mib && 4 * positions > (narrow ? 1 : 3) * n_rows &&
      (narrow || bytes < 20 * mib || positions < 8 * n_rows))
    return 0;
  return positions <= 24 * n_rows;
}

/* Launches in a row that have to find the sparse elements' maximum twice the dense bound before a sequence begins: at
 * first, and at most (twice as many each time a sequence ended because one of its launches did not). A launch that cannot
 * tell max|ds| goes over the matrix twice (at K = 400 on a corpus of 10 M tokens with larger synapses, where the dense elements
 * decide in half of the steps, a step took 61 us so and 54 with every row updated). With the rule, synapses of 1 to 40 times the usual
 * size (the bound grows with their square) at K = 400: 44.5 us up to 2.7 times, 49.6 at 2.9, 50.9 to 51.8 from 3.1 on, every row 51.9. */
#define FV_ROWS_CLEAR 3u
#define FV_ROWS_CLEAR_MOST 1024u
static inline uint32_t fv_rows_clear_after(uint32_t clear) {
  return clear < FV_ROWS_CLEAR_MOST / 2 ? 2 * clear : FV_ROWS_CLEAR_MOST;
}

/* Steps whose xx is kept (a power of two): what fits the dense launch's LDS beside its lists. */
static inline uint32_t fv_rows_age(uint32_t ldk) { return ldk <= 1024 ? 16u : 8u; }
