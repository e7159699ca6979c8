// Large transfers between the device and ordinary (pageable) host memory.
//
// The runtime copies such memory through a staging buffer of its own with one thread: 10 to 17 GB/s, and the caller's
// fresh pages are touched for the first time by that thread, against some 55 GB/s of the link. Here a few host
// threads move pieces between the caller's memory and page-locked slots while the device fills or empties the other
// slots. fv_host_plan.h says from which sizes on that is the faster way.
#pragma once

#include <string.h>

#include <atomic>
#include <memory>
#include <thread>
#include <vector>

#include "fv_host_plan.h"
#include "fv_internal.h"

// Ordinary (pageable) host memory, which the device cannot reach by DMA? (fv_runtime.hip)
bool fv_is_pageable(const void *p);

// Host threads that copy pieces for the length of one call. Pieces are published in order; every thread copies its
// share of every piece. The threads begin with start(), or with the first piece: starting them takes 70 to 100 us, which
// a caller whose pieces come from the device spends while the first one is on its way (20000 targets 402 -> 349 us, 100003
// windows 1615 -> 1533 with four threads).
struct fv_copy_ring {
  struct item {  // `rows` rows of `bytes` bytes
    const char *src;
    char *dst;
    size_t bytes, src_stride, dst_stride;
    uint64_t rows;
  };
  std::vector<item> items;
  std::unique_ptr<std::atomic<uint32_t>[]> finished;  // threads done with item i
  std::atomic<uint32_t> published{0};
  std::atomic<bool> quit{false};
  std::vector<std::thread> workers;
  bool begun = false;
  uint32_t crew = 0;  // threads that started (none: publish copies by itself)

  explicit fv_copy_ring(size_t max_items) : items(max_items), finished(new std::atomic<uint32_t>[max_items]) {
    for (size_t i = 0; i < max_items; ++i) finished[i].store(0);
  }
  void start() {
    if (begun) return;
    begun = true;
    std::atomic<uint32_t> *go = &started;
    try {
      for (uint32_t p = 0; p < FV_COPY_THREADS; ++p) {
        workers.emplace_back([this, p, go] {
          while (go->load(std::memory_order_acquire) == 0) std::this_thread::yield();
          run(p);
        });
        crew++;
      }
    } catch (...) {  // as many threads as the system gives
    }
    started.store(1, std::memory_order_release);  // from here on `crew` does not change
  }
  static void copy_share(const item &it, uint32_t p, uint32_t of) {
    const size_t lo = it.bytes / of * p, hi = p + 1 == of ? it.bytes : it.bytes / of * (p + 1);
    if (hi > lo)
      for (uint64_t r = 0; r < it.rows; ++r) memcpy(it.dst + r * it.dst_stride + lo, it.src + r * it.src_stride + lo, hi - lo);
  }
  void run(uint32_t p) {
    for (uint32_t i = 0;; ++i) {
      while (published.load(std::memory_order_acquire) <= i) {
        if (quit.load(std::memory_order_acquire)) return;
        std::this_thread::yield();
      }
      copy_share(items[i], p, crew);
      finished[i].fetch_add(1, std::memory_order_release);
    }
  }
  uint32_t publish(const item &it) {
    start();
    const uint32_t i = published.load(std::memory_order_relaxed);
    items[i] = it;
    if (crew == 0) copy_share(it, 0, 1);
    published.store(i + 1, std::memory_order_release);
    return i;
  }
  uint32_t publish(const char *src, char *dst, size_t bytes) { return publish(item{src, dst, bytes, bytes, bytes, 1}); }
  void wait(uint32_t i) {
    while (finished[i].load(std::memory_order_acquire) < crew) std::this_thread::yield();
  }
  ~fv_copy_ring() {
    for (uint32_t i = 0; i < published.load(); ++i) wait(i);
    quit.store(true, std::memory_order_release);
    for (auto &t : workers) t.join();
  }

 private:
  std::atomic<uint32_t> started{0};
};

// Page-locked slots of FV_STAGE_SLOT_BYTES, borrowed from the process's pool for the length of one transfer and returned by
// the destructor: n of up to FV_STAGE_SLOTS_LEASED wanted, at least one (waits while other threads hold all of them) unless the
// system gives no page-locked memory or the pool may hold none; the transfer then goes the runtime's way. `events`:
// one per slot.
struct fv_stage_lease {
  char *slots[FV_STAGE_SLOTS_LEASED];
  hipEvent_t events[FV_STAGE_SLOTS_LEASED];
  unsigned n = 0;
  explicit fv_stage_lease(unsigned want);
  ~fv_stage_lease();
  fv_stage_lease(const fv_stage_lease &) = delete;
  fv_stage_lease &operator=(const fv_stage_lease &) = delete;
};

// A stream of the current device, borrowed from the process's pool for the length of one call, which leaves it idle.
// (Making a stream takes up to 4 ms while the process has few.)
struct fv_stream_lease {
  hipStream_t stream = nullptr;
  int device = 0;
  int take(bool make);  // an idle one; if there is none and `make`, a new one, else none. Once per object.
  fv_stream_lease() = default;
  ~fv_stream_lease();
  fv_stream_lease(const fv_stream_lease &) = delete;
  fv_stream_lease &operator=(const fv_stream_lease &) = delete;
};

// Host memory -> device in n_pieces through the lease's slots: piece(t, slot) says what to copy into the slot, consume(t, slot) enqueues the device's
// reading of it on `stream`. Returns when everything has been enqueued and the slots have been read.
template <typename Piece, typename Consume>
int fv_pipe_up(fv_stage_lease &lease, uint64_t n_pieces, hipStream_t stream, Piece piece, Consume consume) {
  const uint64_t S = lease.n;
  if (n_pieces == 1) {
    const fv_copy_ring::item it = piece(0, lease.slots[0]);
    fv_copy_ring::copy_share(it, 0, 1);
    FV_TRY(consume(0, lease.slots[0]));
    FV_HIP(hipStreamSynchronize(stream));
    return FV_OK;
  }
  fv_copy_ring ring(n_pieces);
  int rc = FV_OK;
  for (uint64_t t = 0; t < n_pieces + S - 1 && rc == FV_OK; ++t) {
    if (t < n_pieces) {
      hipError_t e = hipSuccess;
      if (t >= S) e = hipEventSynchronize(lease.events[t % S]);
      if (e != hipSuccess) rc = fv_fail(FV_ERR_HIP, "staged upload failed: %s", hipGetErrorString(e));
      if (rc == FV_OK) ring.publish(piece(t, lease.slots[t % S]));
    }
    if (rc == FV_OK && t + 1 >= S) {
      const uint64_t u = t + 1 - S;
      ring.wait((uint32_t)u);
      rc = consume(u, lease.slots[u % S]);
      if (rc == FV_OK && hipEventRecord(lease.events[u % S], stream) != hipSuccess)
        rc = fv_fail(FV_ERR_HIP, "staged upload: event record failed");
    }
  }
  const hipError_t e = hipStreamSynchronize(stream);  // before the slots go back
  if (rc == FV_OK && e != hipSuccess) rc = fv_fail(FV_ERR_HIP, "staged upload failed: %s", hipGetErrorString(e));
  return rc;
}

// Device -> host memory in n_pieces through the lease's slots: produce(t, slot) enqueues the device's writing of the slot on `stream`, piece(t, slot)
// says where its contents go. Returns when the host memory holds everything.
template <typename Produce, typename Piece>
int fv_pipe_down(fv_stage_lease &lease, uint64_t n_pieces, hipStream_t stream, Produce produce, Piece piece) {
  const uint64_t S = lease.n;
  if (n_pieces == 1) {
    FV_TRY(produce(0, lease.slots[0]));
    FV_HIP(hipStreamSynchronize(stream));
    const fv_copy_ring::item it = piece(0, lease.slots[0]);
    fv_copy_ring::copy_share(it, 0, 1);
    return FV_OK;
  }
  fv_copy_ring ring(n_pieces);
  const uint64_t ahead = S > 1 ? S - 1 : 1;  // pieces the device may be ahead of the host threads by
  int rc = FV_OK;
  for (uint64_t t = 0; t < n_pieces + ahead && rc == FV_OK; ++t) {
    if (t >= ahead) {  // the oldest piece in flight goes to the host threads
      const uint64_t u = t - ahead;
      const hipError_t e = hipEventSynchronize(lease.events[u % S]);
      if (e != hipSuccess) rc = fv_fail(FV_ERR_HIP, "staged download failed: %s", hipGetErrorString(e));
      if (rc == FV_OK) ring.publish(piece(u, lease.slots[u % S]));
    }
    if (rc == FV_OK && t < n_pieces) {
      if (t >= S) ring.wait((uint32_t)(t - S));
      rc = produce(t, lease.slots[t % S]);
      if (rc == FV_OK && hipEventRecord(lease.events[t % S], stream) != hipSuccess)
        rc = fv_fail(FV_ERR_HIP, "staged download: event record failed");
      ring.start();
    }
  }
  (void)hipStreamSynchronize(stream);  // before the slots go back (an error is in rc already)
  return rc;
}

// Plain copies. Page-locked memory and sizes below fv_host_plan.h's go through the runtime. Upwards the caller waits for the stream before
// its own caller may change the source; downwards the host memory is filled on return.
int fv_copy_up(void *dst_dev, const void *src_host, size_t bytes, hipStream_t stream);
int fv_copy_down(void *dst_host, const void *src_dev, size_t bytes, hipStream_t stream);
