// The dense launch that visits only the rows of the matrix somebody needs (device code of fv_train.hip).
//
// Row i of the token-major matrix is read by a step only if token i stands in one of its windows. The dense update
// of any other row (W += s * (-xx[h] * W), element by element) can wait: applied later, one step's update after
// the other, the same fp32 operations run in the same order on the same values, so the matrix comes out the
// same bit for bit. What has to be kept of a step is xx (ldk floats) and s, for 16 steps, or 8 of the widest rows (fv_rows_age). A dense
// launch then visits
//   - the rows its own step has touched (they hold the sentinels of its sparse elements),
//   - the rows the next step reads,
//   - the rows that lack as many steps' updates as are kept,
// and brings them all up to date; the others it neither reads nor writes. At K = 400, V = 20000, w = 11, B = 10000 and
// Zipf-distributed tokens that is half the rows, at K = 1000, V = 50000, w = 15, B = 50000 0.69 of them.
// Measured, every row against rows as needed: the dense launch 21.7 and 17.2 us, 148 and 112; a step of an epoch 52.7 and
// 45.0, 441 and 400; 27.7 and 26.5 at K = 209, V = 7919, w = 7, B = 3001 (fv_rows_pay has more).
//
// What bounds the launch at K = 400 (clock from its first wave; 17.2 us in the trace): arguments, then the list, then the
// first groups of W, one trip behind the other (4.1 us until the block's barrier), 3.7 us for the rows that lack one
// update, 1.5 for those that lack more, 1.1 for the sentinels' records, 4 for the launch itself and its end. Groups in
// flight per thread: 2, 3, 4, 6, 8 measured 17.3, 17.4, 17.2, 17.8, 18.2; two blocks per compute unit (64 registers) 25.9.
// With more streams than one block's the memory does worse at K = 1000 as well (190 against 112).
//
// Which rows: the launch of step t samples the minibatch of step t + 2 and leaves that number in row_need[] of every
// row in it; blocks behind the others of the sparse launch of step t + 1 read row_need[] and row_last[] (the first
// step whose update a row lacks) and write the list the dense launch of step t + 1 works through.
//
// max|ds|: no dense |ds| of neuron h exceeds |xx[h]| * (the largest |W[h][i]| when that was last known + the steps
// since then x |eps|, what a step changes an element by at most). Where the largest |ds| of the sparse elements
// is no less than that bound for every neuron, it is max|ds|. (The ratio of bound and maximum was measured at 0.02 to
// 0.29 at the sizes named above with normal synapses of the size the tests use; it grows with the square of theirs.)
// Otherwise the launch brings every row up to date, takes the maximum over the matrix
// with an exchange between its blocks, and updates every row.
#pragma once

#include "fv_rows_plan.h"
#include "fv_train_dense.h"
#include "fv_train_row_list.h"

#ifndef FV_ROWS_DEPTH
#define FV_ROWS_DEPTH 4  // 16-byte groups of W a thread has in flight
#endif
#ifndef FV_ROWS_LATE
#define FV_ROWS_LATE 2  // and of the rows that lack earlier steps' updates
#endif

// Steps that must follow each other for a sequence to begin, and after how many the bound of |W| starts afresh.
#define FV_ROWS_SEQUENCE 8u
#define FV_ROWS_REFRESH 128u
#define FV_ROWS_DRIFT 0.02  // or when |W| may have grown by this much, which takes at least FV_ROWS_DRIFT_STEPS steps
#define FV_ROWS_DRIFT_STEPS 32

struct fv_rows_args {
  fv_rows_list_args list;
  const float *hist_xx;  // [age][ldk]: xx of step t at t mod age
  float *hist_s;         // [age]: s of step t at t mod age
  uint32_t pieces, piece_magic;  // pieces of 64 groups of a row; 2^32 / pieces + 1 for more than one
  uint32_t rows_per_round;  // rows a block takes at a time (active / ldk4)
  float drift;           // what |W| may have grown by since row_top2 was taken
  uint32_t wave_hits;    // sentinels a wave notes in LDS
};

// The samplers of minibatches to come also say which rows they will read.
__device__ __forceinline__ void fv_rows_mark(uint32_t *need, int32_t column, uint32_t step) {
  if (column >= 0) need[column] = step;
}

// The first step of a sequence: the minibatches of that step and, in a second launch (of the two numbers a row may be
// given the larger has to stay), of the next are sampled and marked here.
struct fv_rows_start_args {
  const int32_t *corpus;
  const uint64_t *pstart;
  int32_t *idx;
  uint64_t first;
  uint32_t n, step, stride, w, V;
  uint32_t *need;
  unsigned long long *count;
};
__global__ __launch_bounds__(256) void fv_rows_start_kernel(fv_rows_start_args a) {
  if (blockIdx.x == 0 && threadIdx.x < 2) a.count[threadIdx.x] = 0;
  const uint32_t entries = a.n * a.stride;
  for (uint32_t e = blockIdx.x * 256 + threadIdx.x; e < entries; e += gridDim.x * 256) {
    const uint32_t r = e / a.stride, c = e - r * a.stride;
    const int32_t col = c < a.w ? fv_column_index(a.corpus[a.pstart[a.first + r] + c], c, a.w, a.V) : -1;
    a.idx[e] = col;
    fv_rows_mark(a.need, col, a.step);
  }
}

// One step's dense update of four elements (fv_apply_four without its report, in five instructions an element). An
// element that does not move has -0 added: that leaves every number as it is, -0 included. A NaN comes out quieted:
// the caller keeps the bits of a sentinel.
__device__ __forceinline__ float fv_rows_apply(float w, float x, float s, float cut) {
  float d = __fmul_rn(s, __fmul_rn(-x, w));
  d = fabsf(d) > cut ? d : -0.0f;
  return __fadd_rn(w, d);
}
__device__ __forceinline__ float4 fv_rows_apply_four(const float4 &w, const float4 &x, float s, float cut) {
  return make_float4(fv_rows_apply(w.x, x.x, s, cut), fv_rows_apply(w.y, x.y, s, cut), fv_rows_apply(w.z, x.z, s, cut),
                     fv_rows_apply(w.w, x.w, s, cut));
}

// `v`, but the bits of `before` where that holds a NaN.
__device__ __forceinline__ float4 fv_rows_keep_nan(const float4 &v, const float4 &before) {
  return make_float4(before.x == before.x ? v.x : before.x, before.y == before.y ? v.y : before.y,
                     before.z == before.z ? v.z : before.z, before.w == before.w ? v.w : before.w);
}

// The updates of the n steps before `step` that a group of four elements lacks (0: none), oldest first; x4 holds the kept
// xx of all steps in LDS, the group is number q of its row, lane i < age of the wave holds the s kept at place i. Lanes
// of a wave may lack different numbers of updates: an update with s = 0 changes nothing. Two steps per turn, so that
// their xx travel together.
__device__ __forceinline__ float4 fv_rows_catch_up(float4 v, uint32_t n, uint32_t step, uint32_t age, const float4 *x4,
                                                   float s_kept, uint32_t ldk4, uint32_t q, float cut) {
  if (!__any(n != 0)) return v;
  const float4 before = v;
  for (uint32_t j = (fv_wave_max_u32(n) + 1u) & ~1u; j != 0; j -= 2) {
    const uint32_t at0 = (step - j) & (age - 1u), at1 = (at0 + 1u) & (age - 1u);
    const float4 xa = x4[at0 * ldk4 + q], xb = x4[at1 * ldk4 + q];
    const float sa = __uint_as_float(fv_readlane(__float_as_uint(s_kept), (int)at0));
    const float sb = __uint_as_float(fv_readlane(__float_as_uint(s_kept), (int)at1));
    v = fv_rows_apply_four(v, xa, j <= n ? sa : 0.0f, cut);
    v = fv_rows_apply_four(v, xb, j - 1u <= n ? sb : 0.0f, cut);
  }
  return fv_rows_keep_nan(v, before);
}

// A sentinel met, as a wave notes it: the record's number (23 bits), the row (27) and the neuron (11) in two words.
__device__ __forceinline__ uint2 fv_rows_hit(float bits, uint32_t row, uint32_t h) {
  return make_uint2((__float_as_uint(bits) & FV_SENTINEL_MAX) | (h << 23), row | ((h >> 9) << FV_ROWS_BITS));
}

// The sentinels of a list of n, dealt over the 64 lanes of a wave, four records in flight per lane
// (fv_finish_sparse_elements without the shares of the rows' largest weights).
__device__ __forceinline__ void fv_rows_finish(const fv_dense_args &a, const uint2 *list, uint32_t n, uint32_t lane, float s,
                                               bool ok) {
  for (uint32_t i0 = 0; i0 < n; i0 += 256) {
    uint32_t p[4];
    fv_slot sl[4];
    bool mine[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t i = i0 + lane + 64u * u;
      const uint2 hit = list[min(i, n - 1)];
      const uint32_t number = (hit.x & FV_SENTINEL_MAX) - 1u, row = hit.y & FV_ROWS_MASK;
      const uint32_t h = (hit.x >> 23) | ((hit.y >> FV_ROWS_BITS) << 9);
      p[u] = row * a.ldk + h;
      mine[u] = i < n && number < a.n_slots;  // a NaN of another origin stays what it is
      const uint64_t at = a.slot_region ? fv_slot_place((h << FV_NB_CLASS_SHIFT) | (row & (FV_NB_CLASSES - 1)), number,
                                                        a.slot_region, a.K * FV_NB_CLASSES)
                                        : number;
      sl[u] = a.slots[mine[u] ? at : 0];
    }
    // the groups' own stores, which put the sentinels back as they came, are over before an element is written
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (mine[u] && sl[u].p == p[u]) ((float *)a.Wt4)[p[u]] = fv_slot_final(sl[u], s, ok, a.update_cut);
    }
  }
}

template <int D, int L>
__global__ __launch_bounds__(FV_ONEPASS_THREADS) void fv_dense_rows_kernel(fv_dense_args a, fv_rows_args b) {
  constexpr uint32_t T = FV_ONEPASS_THREADS;
  extern __shared__ float4 dyn4[];
  float4 *x4 = dyn4;                               // xx of the last steps, age x ldk4 groups
  uint2 *hit_list = (uint2 *)(x4 + b.list.age * a.ldk4);  // the sentinels met, wave_hits of them per wave
  __shared__ uint32_t red2[T / 64][2];
  __shared__ float smem16[16];
  __shared__ float sh_s;
  __shared__ uint32_t sh_ok;
  // every argument in front of the first load of W is asked for here, together (fetched where it is first used, each
  // stood as a trip of its own in the chain)
  asm volatile("" ::"s"(a.Wt4), "s"(a.xx), "s"(a.bmax), "s"(a.scalars), "s"(a.ldk4), "s"(a.K), "s"(a.pstart), "s"(a.ahead_first),
               "s"(a.ahead_n), "s"(a.idx_stride), "s"(a.sparse_base), "s"(a.active), "s"(a.row_top2), "s"(b.list.list),
               "s"(b.list.count), "s"(b.pieces), "s"(b.piece_magic), "s"(b.list.cap), "s"(b.list.n_dense), "s"(b.list.step), "s"(b.hist_xx), "s"(b.hist_s),
               "s"(b.list.age), "s"(b.rows_per_round));
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  uint2 *wave_list = hit_list + (tid >> 6) * b.wave_hits;
  const bool active = tid < a.active;
  const uint32_t q = tid % a.ldk4, r = tid / a.ldk4;
  const uint32_t rows_per_round = b.rows_per_round;
  const uint32_t step = b.list.step, here = step & (b.list.age - 1u);
  // The thread's entries of the block's list first (the list is full of row numbers, also behind its end, so an entry
  // that turns out to lie there is read and not used), then the small loads, then its groups of W.
  const uint32_t *mine = b.list.list + (uint64_t)blockIdx.x * b.list.cap;
  uint32_t cur[D], nxt[D];
  uint32_t parity = step & 1u;
  asm("" : "+v"(parity));  // (a vector load, in the order of the others, not a scalar one waited for by itself)
  const unsigned long long listed_vec = b.list.count[parity];
#pragma unroll
  for (int u = 0; u < D; ++u) cur[u] = mine[min(r + u * rows_per_round, b.list.cap - 1)];
  // The rows that lack earlier steps' updates are taken by waves, a piece of up to 64 groups at a time, so that all lanes of
  // a wave lack the same updates (in waves that hold parts of two rows that work took four times as long): the wave's first
  // pieces.
  constexpr uint32_t WAVES = T / 64;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t *late = mine + (uint64_t)b.list.n_dense * b.list.cap;
  auto late_row = [&](uint32_t i) { return b.pieces == 1 ? i : __umulhi(i, b.piece_magic); };  // i / pieces (i < 2^28)
  uint32_t late_entry[L];
#pragma unroll
  for (int u = 0; u < L; ++u) late_entry[u] = late[min(late_row(wave + u * WAVES), b.list.cap - 1)];
  // the minibatch of the step after the next: the window starts in front of the groups of W, the tokens
  // in front of the stream (a token asked for behind W would wait for all of it)
  constexpr uint32_t TS = T - 64;
  const uint32_t ahead_entries = a.ahead_n * a.idx_stride;
  const uint32_t e0 = blockIdx.x * TS + (tid - 64);
  const bool samples0 = tid >= 64 && e0 < ahead_entries;
  const uint32_t er0 = samples0 ? e0 / a.idx_stride : 0u;
  const uint64_t start0 = a.ahead_n ? a.pstart[a.ahead_first + er0] : 0ull;
  float xh[2], top[2];
  float4 smx[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t h = min(tid + T * j, a.K - 1);
    xh[j] = a.xx[h];
    top[j] = a.row_top2[h].x;
    smx[j] = ((const float4 *)(a.bmax + a.sparse_base))[h];
  }
  const float s_kept = b.hist_s[tid & (b.list.age - 1u)];
  const bool dead = a.scalars[1] != 0.0f;
  const uint2 verdict_before = *(const uint2 *)(a.scalars + 10);
  const uint32_t n_hist = b.list.age * a.ldk4;  // at most 4 T
  const float4 *hist = (const float4 *)b.hist_xx;
  const float4 hist0 = hist[min(tid, n_hist - 1)], hist1 = hist[min(tid + T, n_hist - 1)];
  const float4 hist2 = hist[min(tid + 2 * T, n_hist - 1)], hist3 = hist[min(tid + 3 * T, n_hist - 1)];
  __builtin_amdgcn_sched_barrier(0);
  const uint32_t n_listed = __builtin_amdgcn_readfirstlane((uint32_t)listed_vec);
  const uint32_t n_late = __builtin_amdgcn_readfirstlane((uint32_t)(listed_vec >> 32));
  // entry k of the block's part is number blockIdx.x + k n_dense of the list
  auto listed = [&](uint32_t k) { return blockIdx.x + k * b.list.n_dense < n_listed; };
  float4 w[D];
#pragma unroll
  for (int u = 0; u < D; ++u)
    if (listed(u * rows_per_round)) w[u] = a.Wt4[cur[u] * a.ldk4 + q];
  // piece i of the block's late rows: row late[i / pieces], groups from 64 (i mod pieces) on
  auto late_group = [&](uint32_t i) { return (i - late_row(i) * b.pieces) * 64u + lane; };
  auto late_listed = [&](uint32_t i) { return blockIdx.x + late_row(i) * b.list.n_dense < n_late; };
  float4 lw[L];
#pragma unroll
  for (int u = 0; u < L; ++u)
    if (late_listed(wave + u * WAVES)) lw[u] = a.Wt4[(late_entry[u] & FV_ROWS_MASK) * a.ldk4 + min(late_group(wave + u * WAVES), a.ldk4 - 1)];
  __builtin_amdgcn_sched_barrier(0);

  uint32_t S = 0, F = 0;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (tid + T * j < a.K) {
      // (rounding included: |W| grows by no more than |eps| (1 + 2^-20) and a rounding a step, over at most a few hundred)
      const float bound = __fmul_rn(__fadd_rn(top[j], b.drift), 1.0001f);
      F = max(F, __float_as_uint(__fmul_rn(fabsf(xh[j]), bound)));
      S = max(S, __float_as_uint(fmaxf(fmaxf(smx[j].x, smx[j].y), fmaxf(smx[j].z, smx[j].w))));
    }
  }
  if (tid < n_hist) x4[tid] = hist0;
  if (tid + T < n_hist) x4[tid + T] = hist1;
  if (tid + 2 * T < n_hist) x4[tid + 2 * T] = hist2;
  if (tid + 3 * T < n_hist) x4[tid + 3 * T] = hist3;
  {
    const uint32_t ws = fv_wave_max_u32(S), wf = fv_wave_max_u32(F);
    if (lane == 0) {
      red2[tid >> 6][0] = ws;
      red2[tid >> 6][1] = wf;
    }
  }
  // (LDS only: the groups of W are on their way)
  fv_lds_barrier();
  S = F = 0;
#pragma unroll
  for (uint32_t i = 0; i < T / 64; ++i) {
    S = max(S, red2[i][0]);
    F = max(F, red2[i][1]);
  }
  const float4 xq = x4[here * a.ldk4 + q];
  if (blockIdx.x == 0 && tid == 0) fv_leave_verdict(a, verdict_before, true, !dead && fv_clearly_sparse(S, F));

  float s;
  bool ok = true;
  uint32_t n_hits = 0;  // sentinels the wave has noted (the same in all its lanes)
  // This step's update of a group that is up to date to the steps before it. Sentinels go back as they came and to the
  // wave's list; the bits of those that find it full are returned.
  auto finish_group = [&](float4 v, uint32_t row, bool real, float s, bool ok) -> uint32_t {
    const float4 o = fv_rows_apply_four(v, xq, s, a.update_cut);
    const bool nx = v.x != v.x, ny = v.y != v.y, nz = v.z != v.z, nw = v.w != v.w;
    if (real && ok) a.Wt4[row * a.ldk4 + q] = make_float4(nx ? v.x : o.x, ny ? v.y : o.y, nz ? v.z : o.z, nw ? v.w : o.w);
    uint32_t beyond = 0;
    if (__any(real && (nx || ny || nz || nw))) {
#define FV_ROWS_ELEMENT(is_nan, member, k)                                                               \
  {                                                                                                      \
    const uint64_t met = __ballot(real && is_nan);                                                       \
    const uint32_t at = n_hits + __builtin_amdgcn_mbcnt_hi((uint32_t)(met >> 32),                        \
                                                           __builtin_amdgcn_mbcnt_lo((uint32_t)met, 0)); \
    if (real && is_nan) {                                                                                \
      if (at < a.hit_cap)                                                                                \
        wave_list[at] = fv_rows_hit(member, row, 4u * q + k);                                            \
      else                                                                                               \
        beyond |= 1u << k;                                                                               \
    }                                                                                                    \
    n_hits += (uint32_t)__popcll(met);                                                                   \
  }
      FV_ROWS_ELEMENT(nx, v.x, 0)
      FV_ROWS_ELEMENT(ny, v.y, 1)
      FV_ROWS_ELEMENT(nz, v.z, 2)
      FV_ROWS_ELEMENT(nw, v.w, 3)
#undef FV_ROWS_ELEMENT
    }
    return beyond;
  };
  // an element whose sentinel found the wave's list full, from memory, where that still stands
  auto finish_beyond = [&](uint32_t at, float s, bool ok) {
    fv_finish_sparse_element<false>(a, __float_as_uint(((const float *)a.Wt4)[at]), at, s, ok, nullptr, nullptr);
  };

  const uint32_t c0 = e0 - er0 * a.idx_stride;
  int32_t tok0 = -1;
  if (samples0 && c0 < a.w) tok0 = a.corpus[start0 + c0];
  if (dead || F <= S) {
    // max|ds| is the sparse elements' (or the launch leaves the matrix alone, behind one that gave up, and only puts
    // the sentinels' weights back)
    const float nc = __uint_as_float(S);
    s = a.prec > nc ? a.eps / a.prec : a.eps / nc;  // flyvec/src/cuda_funcs.cu:1797-1799
    ok = !dead;
    const uint32_t n_mine = n_listed > blockIdx.x ? min((n_listed - blockIdx.x - 1u) / b.list.n_dense + 1u, b.list.cap) : 0u;
    const uint32_t rounds = (n_mine + rows_per_round - 1) / rows_per_round;
    if (rounds > D) {
#pragma unroll
      for (int u = 0; u < D; ++u) nxt[u] = mine[min(r + (D + u) * rows_per_round, n_mine - 1)];
    }
    static_assert(4 * D <= 64, "one bit per element of a thread");
    for (uint32_t c = 0; c < rounds; c += D) {
      uint64_t beyond = 0;
#pragma unroll
      for (int u = 0; u < D; ++u) {
        if (c + u < rounds) {
          const uint32_t at = r + (c + u) * rows_per_round, entry = cur[u];
          const bool real = active && at < n_mine;
          beyond |= (uint64_t)finish_group(w[u], entry, real, s, ok) << (4 * u);
          if (c + D + u < rounds) {  // the round that takes this one's place (an entry past the end: the last one again)
            cur[u] = nxt[u];
            w[u] = a.Wt4[cur[u] * a.ldk4 + q];
            nxt[u] = mine[min(at + 2 * D * rows_per_round, n_mine - 1)];
          }
        }
      }
      while (beyond) {
        const uint32_t k = (uint32_t)__ffsll((long long)beyond) - 1u;
        beyond &= beyond - 1;
        const uint32_t row = mine[r + (c + (k >> 2)) * rows_per_round];
        finish_beyond(4u * (row * a.ldk4 + q) + (k & 3u), s, ok);
      }
    }
    const uint32_t n_behind = n_late > blockIdx.x ? min((n_late - blockIdx.x - 1u) / b.list.n_dense + 1u, b.list.cap) : 0u;
    if (ok) {
      const uint32_t n_pieces = n_behind * b.pieces;
      for (uint32_t i0 = wave; i0 < n_pieces; i0 += L * WAVES) {
#pragma unroll
        for (int u = 0; u < L; ++u) {
          const uint32_t i = i0 + u * WAVES;
          if (i < n_pieces) {
            const uint32_t entry = __builtin_amdgcn_readfirstlane(late_entry[u]), at_g = late_group(i), g = min(at_g, a.ldk4 - 1);
            float4 v = lw[u];
            for (uint32_t j = entry >> FV_ROWS_BITS; j != 0; --j) {
              const uint32_t at = (step - j) & (b.list.age - 1u);
              v = fv_rows_apply_four(v, x4[at * a.ldk4 + g], __uint_as_float(fv_readlane(__float_as_uint(s_kept), (int)at)), a.update_cut);
            }
            v = fv_rows_apply_four(v, x4[here * a.ldk4 + g], s, a.update_cut);
            if (at_g < a.ldk4)
              a.Wt4[(entry & FV_ROWS_MASK) * a.ldk4 + g] = fv_rows_keep_nan(v, lw[u]);
          }
          const uint32_t in = i + L * WAVES;  // the piece that takes this one's place
          if (in < n_pieces) {
            late_entry[u] = late[late_row(in)];
            lw[u] = a.Wt4[(late_entry[u] & FV_ROWS_MASK) * a.ldk4 + min(late_group(in), a.ldk4 - 1)];
          }
        }
      }
      for (uint32_t i = tid; i < n_mine; i += T) b.list.last[mine[i]] = step + 1u;
      for (uint32_t i = tid; i < n_behind; i += T) b.list.last[late[i] & FV_ROWS_MASK] = step + 1u;
    }
    if (blockIdx.x == 0 && tid == 0) {
      if (ok) {
        a.scalars[0] = nc;
        a.path_count[0] += 1;
        b.hist_s[here] = s;
      }
      b.list.count[(step + 1u) & 1u] = 0;  // for the next step's list
    }
  } else {
    // Every row: what it lacks first, and the maximum over what the matrix then is; then this step's update.
    const uint32_t row0 = blockIdx.x + b.list.n_dense * r, row_step = b.list.n_dense * rows_per_round;
    const uint32_t all_rounds = (a.n_rows + row_step - 1) / row_step;
    float m = __uint_as_float(S);
    for (uint32_t c = 0; c < all_rounds; ++c) {
      const uint32_t row = row0 + c * row_step;
      const bool real = active && row < a.n_rows;
      const uint32_t p4 = (real ? row : 0u) * a.ldk4 + q;
      const uint32_t lacks = real ? step - max(b.list.last[row], b.list.first) : 0u;
      // (a row with sentinels is up to date)
      const float4 v = fv_rows_catch_up(a.Wt4[p4], lacks, step, b.list.age, x4, s_kept, a.ldk4, q, a.update_cut);
      if (lacks) a.Wt4[p4] = v;
      if (real) m = fv_absmax_four(m, xq, v);
    }
    fv_onepass_exchange(a, m, a.spin_limit, false, smem16, &sh_s, &sh_ok);
    __syncthreads();
    ok = sh_ok != 0;
    s = sh_s;
    if (blockIdx.x == 0 && tid == 0) {
      b.hist_s[here] = s;
      b.list.count[(step + 1u) & 1u] = 0;
    }
    for (uint32_t c = 0; c < all_rounds; ++c) {
      const uint32_t row = row0 + c * row_step;
      const bool real = active && row < a.n_rows;
      const uint32_t p4 = (real ? row : 0u) * a.ldk4 + q;
      for (uint32_t beyond = finish_group(a.Wt4[p4], row, real, s, ok); beyond; beyond &= beyond - 1)
        finish_beyond(4u * p4 + (uint32_t)__ffs((int)beyond) - 1u, s, ok);
      if (real && q == 0) b.list.last[row] = ok ? step + 1u : step;
    }
  }
  if (samples0) {
    const int32_t col = c0 < a.w ? fv_column_index(tok0, c0, a.w, a.V) : -1;
    a.idx_ahead[e0] = col;
    fv_rows_mark(b.list.need, col, step + 2u);
  }
  if (tid >= 64) {
    // (a minibatch with more positions than the launch has sampling threads: four at a time)
    const uint32_t hop = b.list.n_dense * TS;
    for (uint32_t e = e0 + hop; e < ahead_entries; e += 4 * hop) {
      uint32_t c[4];
      uint64_t at[4];
      int32_t tok[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t ek = e + k * hop < ahead_entries ? e + k * hop : e;
        const uint32_t rr = ek / a.idx_stride;
        c[k] = ek - rr * a.idx_stride;
        at[k] = a.pstart[a.ahead_first + rr];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) tok[k] = a.corpus[at[k] + (c[k] < a.w ? c[k] : 0u)];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (e + k * hop < ahead_entries) {
          const int32_t col = c[k] < a.w ? fv_column_index(tok[k], c[k], a.w, a.V) : -1;
          a.idx_ahead[e + k * hop] = col;
          fv_rows_mark(b.list.need, col, step + 2u);
        }
    }
  }
  // the sentinels the wave has met, dealt over its lanes
  fv_rows_finish(a, wave_list, min(n_hits, a.hit_cap), lane, s, ok);
}

// Every row brought up to date to the steps before `step`, and every block's share of the rows' two largest weights
// left as a dense launch leaves them: behind the last step of a sequence, and now and then inside one, so that the
// bound of |W| starts afresh. Behind a launch that gave up no row lacks an update (that launch has left every row as
// the step before it did, and the steps enqueued behind it change nothing): the shares only.
#ifndef FV_ROWS_SETTLE_DEPTH
#define FV_ROWS_SETTLE_DEPTH 4
#endif
__global__ __launch_bounds__(FV_ONEPASS_THREADS) void fv_rows_settle_kernel(fv_dense_args a, fv_rows_args b) {
  constexpr uint32_t T = FV_ONEPASS_THREADS;
  constexpr int D = FV_ROWS_SETTLE_DEPTH;
  extern __shared__ float4 dyn4[];
  float4 *x4 = dyn4;
  float2 *pairs = (float2 *)(x4 + b.list.age * a.ldk4);
  const uint32_t tid = threadIdx.x;
  const bool dead = a.scalars[1] != 0.0f;
  const bool active = tid < a.active;
  const uint32_t q = tid % a.ldk4, r = tid / a.ldk4;
  const uint32_t rows_per_round = a.active / a.ldk4;
  const uint32_t row0 = blockIdx.x + b.list.n_dense * r, row_step = b.list.n_dense * rows_per_round;
  const uint32_t rounds = (a.n_rows + row_step - 1) / row_step;
  const uint32_t row_inside = min(row0, a.n_rows - 1);
  float4 w[D];
  uint32_t last[D];
#pragma unroll
  for (int u = 0; u < D; ++u) {
    const uint32_t row = row0 + u * row_step;
    last[u] = b.list.last[row < a.n_rows ? row : row_inside];
    w[u] = a.Wt4[(row < a.n_rows ? row : row_inside) * a.ldk4 + q];
  }
  for (uint32_t i = tid; i < b.list.age * a.ldk4; i += T) x4[i] = ((const float4 *)b.hist_xx)[i];
  const float s_kept = b.hist_s[tid & (b.list.age - 1u)];
  __syncthreads();
  float t1[4] = {0.0f, 0.0f, 0.0f, 0.0f}, t2[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (uint32_t c = 0; c < rounds; c += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      const uint32_t row = row0 + (c + u) * row_step;
      const bool real = active && row < a.n_rows;
      const uint32_t lacks = real && !dead ? b.list.step - max(last[u], b.list.first) : 0u;
      const float4 v = fv_rows_catch_up(w[u], lacks, b.list.step, b.list.age, x4, s_kept, a.ldk4, q, a.update_cut);
      if (real) {
        if (lacks) a.Wt4[row * a.ldk4 + q] = v;
        fv_top2_insert_four(t1, t2, v, __builtin_isunordered(v.x, v.y) || __builtin_isunordered(v.z, v.w));
      }
      const uint32_t rown = row + D * row_step;
      last[u] = b.list.last[rown < a.n_rows ? rown : row_inside];
      w[u] = a.Wt4[(rown < a.n_rows ? rown : row_inside) * a.ldk4 + q];
    }
  }
  if (active) {
#pragma unroll
    for (int e = 0; e < 4; ++e) pairs[(e * rows_per_round + r) * a.ldk4 + q] = make_float2(t1[e], t2[e]);
  }
  __syncthreads();
  for (uint32_t h = tid; h < a.K; h += T) {
    const uint32_t e = h & 3u, qq = h >> 2;
    float m1 = 0.0f, m2 = 0.0f;
    for (uint32_t rr = 0; rr < rows_per_round; ++rr) {
      const float2 p = pairs[(e * rows_per_round + rr) * a.ldk4 + qq];
      fv_top2_merge(m1, m2, p.x, p.y);
    }
    a.top2_part[(uint64_t)blockIdx.x * a.ldk + h] = make_float2(m1, m2);
  }
}

static int fv_rows_fit(size_t smem, size_t smem_settle) {
  int nb = 0, nb2 = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, (fv_dense_rows_kernel<FV_ROWS_DEPTH, FV_ROWS_LATE>), FV_ONEPASS_THREADS, smem) !=
          hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb2, fv_rows_settle_kernel, FV_ONEPASS_THREADS, smem_settle) !=
          hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return nb >= 1 && nb2 >= 1;
}
