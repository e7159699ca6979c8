/* Host build of flyvec_amd/csrc/fv_window_scan.h for the CPU test-suite. */
#include "fv_window_scan.h"

uint64_t fvt_scan_tiles(uint64_t n_chunks) { return fv_scan_tiles(n_chunks); }
uint64_t fvt_scan_max_tiles(void) { return FV_SCAN_MAX_TILES; }
uint32_t fvt_scan_tile(void) { return FV_SCAN_TILE; }
uint32_t fvt_scan_threads(void) { return FV_SCAN_THREADS; }
uint32_t fvt_scan_parts(void) { return FV_SCAN_PARTS; }
void fvt_scan_grids(uint64_t n_tiles, uint32_t *out) {
  const fv_scan_grid a = fv_scan_totals_grid(n_tiles), b = fv_scan_expand_grid(n_tiles);
  out[0] = a.x;
  out[1] = a.y;
  out[2] = b.x;
  out[3] = b.y;
}
