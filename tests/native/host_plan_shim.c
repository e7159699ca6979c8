/* Host build of flyvec_amd/csrc/fv_host_plan.h for the CPU test-suite. */
#include "fv_host_plan.h"

uint64_t fvt_slot_bytes(void) { return FV_STAGE_SLOT_BYTES; }
int fvt_upload_staged(uint64_t bytes) { return fv_upload_staged(bytes); }
int fvt_download_staged(uint64_t bytes) { return fv_download_staged(bytes); }
int fvt_matrix_upload_staged(uint64_t bytes) { return fv_matrix_upload_staged(bytes); }
uint64_t fvt_copy_pieces(uint64_t bytes) { return fv_copy_pieces(bytes); }
uint64_t fvt_copy_slots(uint64_t bytes) { return fv_copy_slots(bytes); }
uint64_t fvt_copy_piece_bytes(uint64_t bytes, uint64_t t) { return fv_copy_piece_bytes(bytes, t); }
uint64_t fvt_matrix_pieces(uint32_t K, uint64_t N) { return fv_cut_matrix(K, N).n; }
void fvt_matrix_piece(uint32_t K, uint64_t N, uint64_t t, uint64_t *out) {
  const fv_matrix_pieces p = fv_cut_matrix(K, N);
  const fv_matrix_piece m = fv_matrix_piece_at(&p, t);
  out[0] = m.h;
  out[1] = m.rows;
  out[2] = m.i;
  out[3] = m.cols;
  out[4] = m.pitch;
}
void fvt_plan_hash(uint64_t n, uint32_t w, uint64_t bits_row, uint64_t codes_row, int bits_pageable, int codes_pageable,
                   uint64_t *out) {
  const fv_hash_plan p = fv_plan_hash(n, bits_row, codes_row, bits_pageable, codes_pageable);
  out[0] = (uint64_t)fv_hash_is_direct(n, w, bits_row + codes_row);
  out[1] = !out[0] && p.crew;
  out[2] = p.chunk;
}
/* the same with the staging: slots asked for, then places where the pool gives `got` (0: as many) */
void fvt_hash_stage(uint64_t n, uint64_t bits_row, uint64_t codes_row, uint64_t in_row, uint64_t out_row, unsigned got,
                    uint64_t *out) {
  fv_hash_plan p = fv_plan_hash(n, bits_row, codes_row, 1, 1);
  const unsigned want = fv_hash_stage_slots(&p, in_row, out_row), slots = got && got < want ? got : want;
  const fv_hash_staging s = fv_hash_stage(&p, in_row, out_row, slots);
  out[0] = want;
  out[1] = slots;
  out[2] = p.chunk;
  out[3] = (uint64_t)s.lanes;
  for (int l = 0; l < s.lanes; ++l) {
    out[4 + 4 * l] = s.slot[l];
    out[5 + 4 * l] = s.at[l];
    out[6 + 4 * l] = s.in_slot[l];
    out[7 + 4 * l] = s.in_at[l];
  }
}
