// Which way a transfer between the device and ordinary (pageable) host memory goes, and in which pieces: the rules and
// the arithmetic of fv_host_copy.h, shared with the CPU test-suite. Plain C.
//
// The other way is the runtime's copy of such memory, for a matrix with a staging matrix on the device. Both sides
// measured with pauses and new arrays between the calls, as set-up calls come (microseconds, runtime against slots; two
// runs each; back to back the slots do a little better):
//   upload    8 MB 480-560, 590-650;  12 MB 700-850, 810-920;  16 MB on one machine 920-970, 1020-1045, on another 1120-1190,
//             1040-1170;  24 MB 1570-1590, 1515-1660 and 1710-1800, 1490-1530;  32 MB 2030-2120, 1840-1990;  64 MB 4120,
//             3680: the runtime reads the caller's pages at 17 GB/s, four threads at little more
//   download  4 MB 250, 280 (in eight pieces);  5 MB 316-390, 213-242;  8 MB 480-610, 284-316;  16 MB 930-960, 470-505;
//             64 MB 6300, 1950 (the result's pages are touched for the first time, by four threads). In pieces of 512 KB
//             instead of whole slots 8 MB took 480-560 and 14 MB 775-800.
//   matrix up, K = 400: 6 MB 314-337, 314-335, with the hasher around it 368-412, 415-496;  8 MB 376-411, 346-381 and
//             426-471, 432-521;  12 MB 519-530, 442-456 and 558-611, 535-562;  64 MB 2430, 1680 and 2500, 1900.  In one
//             piece: 0.25 MB 52, 50;  1 MB 70-81, 77;  4 MB 232-254, 228
//   matrix down, K = 400: 8 MB 539-560, 320-347;  12 MB 800, 415;  64 MB 6550, 2700.  In one piece: 0.25 MB 56, 47;
//             1 MB 82-87, 81;  4 MB 324-330, 210
// A matrix that fits a slot goes as one piece, moved by the calling thread: cut into tiles of 64 rows, as the larger ones
// are, 1 MB at K = 400 took 235 us, and page-locked four slots for it.
#pragma once

#include <stddef.h>
#include <stdint.h>

#define FV_STAGE_SLOT_BYTES ((size_t)4 << 20)
#define FV_STAGE_SLOTS_MAX 8    /* of the process: 32 MB */
#define FV_STAGE_SLOTS_LEASED 4 /* by one transfer */
#define FV_STAGE_TILE_ROWS 64u  /* of a matrix that goes in several pieces */

#define FV_STAGE_UP_BYTES ((size_t)24 << 20)        /* plain uploads through the slots from here on */
#define FV_STAGE_DOWN_BYTES ((size_t)5 << 20)       /* plain downloads */
#define FV_STAGE_MATRIX_UP_BYTES ((size_t)8 << 20)  /* matrices upwards, and those that fit one slot; downwards all */

static inline int fv_upload_staged(size_t bytes) { return bytes >= FV_STAGE_UP_BYTES; }
static inline int fv_download_staged(size_t bytes) { return bytes >= FV_STAGE_DOWN_BYTES; }
static inline int fv_matrix_upload_staged(size_t bytes) {
  return bytes <= FV_STAGE_SLOT_BYTES || bytes >= FV_STAGE_MATRIX_UP_BYTES;
}

/* Host threads of a transfer, started while its first piece is on its way (fv_copy_ring). Four against six against eight
 * (microseconds): 20000 targets (8 MB) 349, 395, 443;  a corpus with its order and table read back (21 MB) 1531, 1609,
 * 1640;  100003 windows to 40 MB of codes 1533, 1435, 1485;  a matrix of 64 MB up and down 4790, 4590, 4540. Six for the large
 * transfers alone made the first batch of four behind one slower (20000 targets on a new hasher 590 to 730 instead of
 * 490 to 620). */
#define FV_COPY_THREADS 4

/* Pieces of a plain copy: whole slots and a rest. */
static inline uint64_t fv_copy_pieces(size_t bytes) { return (bytes + FV_STAGE_SLOT_BYTES - 1) / FV_STAGE_SLOT_BYTES; }
static inline unsigned fv_copy_slots(size_t bytes) {
  return bytes < FV_STAGE_SLOTS_LEASED * FV_STAGE_SLOT_BYTES ? (unsigned)fv_copy_pieces(bytes) : FV_STAGE_SLOTS_LEASED;
}
static inline size_t fv_copy_piece_bytes(size_t bytes, uint64_t t) {
  const size_t left = bytes - (size_t)t * FV_STAGE_SLOT_BYTES;
  return left < FV_STAGE_SLOT_BYTES ? left : FV_STAGE_SLOT_BYTES;
}

/* Pieces of a K x N row-major matrix of floats: the whole of it as it lies in memory if it fits a slot, else tiles of
 * FV_STAGE_TILE_ROWS rows by as many columns as a slot holds. Piece t: `rows` rows from row `h`, `cols` columns from
 * column `i`, rows of `pitch` floats in the slot. */
typedef struct fv_matrix_pieces {
  uint32_t K;
  uint64_t N, columns, across, n;
} fv_matrix_pieces;

typedef struct fv_matrix_piece {
  uint32_t h, rows;
  uint64_t i, cols, pitch;
} fv_matrix_piece;

static inline fv_matrix_pieces fv_cut_matrix(uint32_t K, uint64_t N) {
  fv_matrix_pieces p;
  p.K = K;
  p.N = N;
  if (N <= FV_STAGE_SLOT_BYTES / sizeof(float) / K) {
    p.columns = N;
    p.across = p.n = 1;
  } else {
    p.columns = FV_STAGE_SLOT_BYTES / (FV_STAGE_TILE_ROWS * sizeof(float));
    p.across = (N + p.columns - 1) / p.columns;
    p.n = p.across * ((K + FV_STAGE_TILE_ROWS - 1) / FV_STAGE_TILE_ROWS);
  }
  return p;
}

static inline unsigned fv_matrix_slots(const fv_matrix_pieces *p) {
  return p->n < FV_STAGE_SLOTS_LEASED ? (unsigned)p->n : FV_STAGE_SLOTS_LEASED;
}

static inline fv_matrix_piece fv_matrix_piece_at(const fv_matrix_pieces *p, uint64_t t) {
  fv_matrix_piece m;
  if (p->n == 1) {
    m.h = 0;
    m.rows = p->K;
    m.i = 0;
    m.cols = m.pitch = p->N;
    return m;
  }
  m.h = (uint32_t)(t / p->across) * FV_STAGE_TILE_ROWS;
  m.rows = p->K - m.h < FV_STAGE_TILE_ROWS ? p->K - m.h : FV_STAGE_TILE_ROWS;
  m.i = t % p->across * p->columns;
  m.cols = p->N - m.i < p->columns ? p->N - m.i : p->columns;
  m.pitch = (m.cols + FV_STAGE_TILE_ROWS - 1) / FV_STAGE_TILE_ROWS * FV_STAGE_TILE_ROWS;
  return m;
}

/* ---- batches of codes from host arrays ---- */

#define FV_HASH_CHUNK (1u << 17) /* most windows per chunk */
#define FV_HASH_LANES 4          /* most chunks in flight */
/* A batch is cut into about this many chunks, of output that takes the link some 30 us or more: one call's copies in,
 * kernel, copies out and host copies then overlap also for batches that fit one chunk. (4 or 16 chunks: the same within
 * the runs' differences, 20000 targets 365 and 339 us, 340 with 8; chunks of 0.75 MB 394, of 3 MB 333, for twice the
 * page-locked memory.) */
#define FV_HASH_CHUNKS 8
#define FV_HASH_CHUNK_MIN_BYTES ((uint64_t)3 << 19)
/* Results of this size and more, for pageable memory, are worth the host threads. */
#define FV_HASH_CREW_BYTES ((uint64_t)4 << 20)
/* Batches whose indices and codes take no more than this go through one page-locked buffer that the kernel itself
 * reads and writes: a launch and a wait, where two copies and their waits took 30 us of 44 (126 KB: 24 us against 82, 252
 * KB: 29 against 49). It is still faster beyond (513 KB: 41 against 54, 1 MB: 66 against 80, 2 MB: 125 against 145);
 * the line lies where it does because every hasher page-locks that much when it is made. */
#define FV_HASH_DIRECT_BYTES ((uint64_t)1 << 18)

static inline int fv_hash_is_direct(uint64_t n, uint32_t w, uint64_t out_row) {
  return n <= FV_HASH_DIRECT_BYTES && n * (w * sizeof(int32_t) + out_row) <= FV_HASH_DIRECT_BYTES;
}

typedef struct fv_hash_plan {
  int crew;       /* host threads and page-locked staging */
  uint64_t chunk; /* windows per chunk */
} fv_hash_plan;

/* The other batches. n windows; bits_row, codes_row: bytes of a window's packed and plain codes, 0 where not asked for.
 * Host threads where results for pageable memory are large, or come in more than FV_HASH_CHUNK windows: there the
 * chunks overlap on two streams, and the runtime's copies of pageable memory, which the host waits for, would take
 * that away (500000 windows to 4 MB of packed codes: 835 us, 1230 with the runtime's copies; 200000 to 3 MB: 580, 640). */
static inline fv_hash_plan fv_plan_hash(uint64_t n, uint64_t bits_row, uint64_t codes_row, int bits_pageable,
                                        int codes_pageable) {
  fv_hash_plan p = {0, FV_HASH_CHUNK};
  const uint64_t out_row = bits_row + codes_row;
  p.crew = ((bits_row && bits_pageable) || (codes_row && codes_pageable)) &&
           (n > FV_HASH_CHUNK || n * out_row >= FV_HASH_CREW_BYTES);
  if (p.crew) {
    const uint64_t share = (n + FV_HASH_CHUNKS - 1) / FV_HASH_CHUNKS, least = FV_HASH_CHUNK_MIN_BYTES / out_row + 1;
    const uint64_t want = share > least ? share : least;
    p.chunk = want < FV_HASH_CHUNK ? want : FV_HASH_CHUNK;
  }
  if (p.chunk > n) p.chunk = n;
  return p;
}

/* The staging of the chunks in flight, in_row bytes of indices and out_row of codes per window (0 where not staged).
 * Light indices (a fourth of the codes and less): four chunks in flight, each in a region of its own for both, and the
 * calling thread copies the indices itself, so that the host threads copy codes all the time (100003 windows of 444 bytes,
 * 40 MB of codes: 1.44 ms, with two chunks and the threads copying both 1.75; 20000 targets 340 us and 376; three chunks in
 * flight are in between). Heavy ones: two chunks in flight, the indices in slots of their own where the chunks are large,
 * so that they may be nearly twice as large (1 M windows of 44 and 56 bytes: 3.46 ms; in the other layout 4.03). */
typedef struct fv_hash_staging {
  int lanes;                      /* chunks in flight */
  int light;                      /* the calling thread copies the indices */
  uint32_t slot[FV_HASH_LANES];   /* that holds the lane's codes */
  size_t at[FV_HASH_LANES];       /* where in the slot they begin */
  uint32_t in_slot[FV_HASH_LANES];/* the same of its indices */
  size_t in_at[FV_HASH_LANES];
} fv_hash_staging;

static inline int fv_hash_indices_light(uint64_t in_row, uint64_t out_row) { return 4 * in_row <= out_row; }

/* Slots that the staging asks the pool for. */
static inline unsigned fv_hash_stage_slots(const fv_hash_plan *p, uint64_t in_row, uint64_t out_row) {
  const uint64_t bytes = p->chunk * (in_row + out_row) + 128;
  if (fv_hash_indices_light(in_row, out_row)) {
    const uint64_t want = (FV_HASH_LANES * bytes + FV_STAGE_SLOT_BYTES - 1) / FV_STAGE_SLOT_BYTES;
    return (unsigned)(want < FV_HASH_LANES ? want : FV_HASH_LANES);
  }
  if (2 * bytes <= FV_STAGE_SLOT_BYTES) return 1;
  return bytes <= FV_STAGE_SLOT_BYTES ? 2 : 4;
}

/* Where the staging lies in the `slots` (1 .. that many) that the pool gave; the chunk shrinks to what they hold. */
static inline fv_hash_staging fv_hash_stage(fv_hash_plan *p, uint64_t in_row, uint64_t out_row, unsigned slots) {
  fv_hash_staging s;
  s.light = fv_hash_indices_light(in_row, out_row);
  s.lanes = s.light ? FV_HASH_LANES : 2;
  const int apart = !s.light && slots >= 4;
  const unsigned per_slot = apart ? 1 : ((unsigned)s.lanes + slots - 1) / slots;
  const size_t region = FV_STAGE_SLOT_BYTES / per_slot & ~(size_t)63;
  const uint64_t widest = !apart ? in_row + out_row : in_row > out_row ? in_row : out_row;
  if (p->chunk > (region - 64) / widest) p->chunk = (region - 64) / widest;
  for (uint32_t l = 0; l < (uint32_t)s.lanes; ++l) {
    s.slot[l] = l / per_slot;
    s.at[l] = l % per_slot * region;
    s.in_slot[l] = apart ? l + 2 : s.slot[l];
    s.in_at[l] = apart ? 0 : s.at[l] + ((p->chunk * out_row + 63) & ~(size_t)63);
  }
  return s;
}
