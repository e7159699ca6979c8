// Tiles and launch shapes of the window scan (flyvec/src/prune_input.cpp:64-122 as data-parallel passes), shared by the
// kernels' host and device code and by the CPU test-suite. Plain C.
//
// The runtime refuses a launch whose blocks times threads reach 2^32 in one dimension. One block per tile in the first
// dimension therefore takes a corpus of up to 2^35 - 4096 chunks, 275 GB of offsets; the expansion's parts of a tile
// lie in the second dimension, so that it takes as many.
#pragma once

#include <stdint.h>

#define FV_SCAN_THREADS 256u
#define FV_SCAN_ITEMS 8u /* chunks per thread */
#define FV_SCAN_TILE (FV_SCAN_THREADS * FV_SCAN_ITEMS)
#define FV_SCAN_PARTS 8u /* blocks of the expansion per tile */
#define FV_SCAN_MAX_TILES (0xffffffffull / FV_SCAN_THREADS)

typedef struct fv_scan_grid {
  uint32_t x, y;
} fv_scan_grid;

static inline uint64_t fv_scan_tiles(uint64_t n_chunks) {
  return n_chunks / FV_SCAN_TILE + (n_chunks % FV_SCAN_TILE != 0);
}

/* Blocks of the tile totals' launch and of the expansion's, for 1 .. FV_SCAN_MAX_TILES tiles. */
static inline fv_scan_grid fv_scan_totals_grid(uint64_t n_tiles) {
  const fv_scan_grid g = {(uint32_t)n_tiles, 1};
  return g;
}

static inline fv_scan_grid fv_scan_expand_grid(uint64_t n_tiles) {
  const fv_scan_grid g = {(uint32_t)n_tiles, FV_SCAN_PARTS};
  return g;
}
