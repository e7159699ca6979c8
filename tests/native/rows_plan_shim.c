/* Host build of flyvec_amd/csrc/fv_rows_plan.h for the CPU test-suite. */
#include "fv_rows_plan.h"

int fvt_rows_pay(uint64_t n_rows, uint32_t ldk, uint64_t positions) { return fv_rows_pay(n_rows, ldk, positions); }
uint32_t fvt_rows_clear_first(void) { return FV_ROWS_CLEAR; }
uint32_t fvt_rows_clear_most(void) { return FV_ROWS_CLEAR_MOST; }
uint32_t fvt_rows_clear_after(uint32_t clear) { return fv_rows_clear_after(clear); }
