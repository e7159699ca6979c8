// Which rows of the matrix a dense launch visits (fv_train_rows.h): listed by blocks behind the others of the sparse
// launch in front of it (device code of fv_train.hip).
#pragma once

#include "fv_train_group.h"

#define FV_ROWS_BITS 27u  // of a list entry: the row; above it the updates of earlier steps that the row lacks
#define FV_ROWS_MASK ((1u << FV_ROWS_BITS) - 1u)

struct fv_rows_list_args {
  uint32_t *need;        // per row: the newest step whose minibatch holds it (filled to a multiple of FV_SP_THREADS)
  uint32_t *last;        // per row: the first step whose update it lacks
  // Two lists, each with a part of `cap` entries for every block of the dense launch: the rows that lack this step's update
  // only, and behind all of those parts the rows that lack earlier steps' as well (they hold no sentinel of this step)
  uint32_t *list;
  unsigned long long *count;  // rows listed, by the parity of the step: in the first list, and in the second << 32
  uint32_t cap, n_dense;      // entries per part, blocks of the dense launch
  uint32_t step, first;       // this step; no row lacks the update of a step before `first`
  uint32_t age;               // steps whose xx and s are kept (a power of two): a row that would lack as many is listed
  uint32_t n_rows;
  const float *dead;      // not 0: a launch has given up; the ones behind it leave the rows as they are
};

// FV_SP_THREADS rows per block, one per thread: those whose tokens stand in this step's minibatch or in the next one's, and
// those that lag too far behind. The parts of a list are filled in turn, so every block of the dense launch gets its
// share whatever rows are listed. One atomic per block; the order of a list is of no consequence.
__device__ __forceinline__ void fv_rows_list_block(const fv_rows_list_args &a, uint32_t block, uint32_t *red /*17*/) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, row = block * FV_SP_THREADS + tid;
  const uint32_t need = a.need[row];
  // updates of steps before this one (behind a launch that gave up there are none, and the rows that hold sentinels have to
  // be in the first list all the same)
  const uint32_t lacks = *a.dead != 0.0f ? 0u : a.step - max(a.last[row], a.first);
  const bool take = row < a.n_rows && (need >= a.step || lacks + 1 >= a.age), late = take && lacks != 0;
  const uint32_t mine = late ? 0x10000u : take ? 1u : 0u;
  const uint32_t incl = fv_wave_inclusive_scan_u32(mine);
  if (lane == 63u) red[tid >> 6] = incl;
  fv_lds_barrier();
  uint32_t before = 0, total = 0;
#pragma unroll
  for (uint32_t i = 0; i < FV_SP_THREADS / 64; ++i) {
    before += i < (tid >> 6) ? red[i] : 0u;
    total += red[i];
  }
  if (tid == 0) {
    const unsigned long long both = (total & 0xffffu) | ((unsigned long long)(total >> 16) << 32);
    const unsigned long long at = both ? atomicAdd(&a.count[a.step & 1u], both) : 0ull;
    red[15] = (uint32_t)at;
    red[16] = (uint32_t)(at >> 32);
  }
  fv_lds_barrier();
  if (take) {
    const uint32_t rank = before + incl - mine, at = late ? red[16] + (rank >> 16) : red[15] + (rank & 0xffffu);
    const uint32_t part = at % a.n_dense + (late ? a.n_dense : 0u), place = at / a.n_dense;
    if (place < a.cap) a.list[(uint64_t)part * a.cap + place] = row | (lacks << FV_ROWS_BITS);
  }
}
static inline uint32_t fv_rows_list_blocks(uint64_t n_rows) { return (uint32_t)((n_rows + FV_SP_THREADS - 1) / FV_SP_THREADS); }
