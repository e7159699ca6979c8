// Runtime plumbing of libflyvec_hip.so: error reporting, device queries, pinned / device
// memory helpers, and the layout change between the checkpoint matrix (K x N row-major) and
// the token-major matrix the kernels read.
#include <string.h>

#include <condition_variable>
#include <mutex>
#include <string>

#include "fv_host_copy.h"

static thread_local std::string g_last_error;

int fv_fail(int code, const char *fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

void fv_clear_error() { g_last_error.clear(); }

extern "C" const char *fv_last_error(void) { return g_last_error.c_str(); }

extern "C" int fv_device_count(int *out_count) {
  FV_REQUIRE(out_count, FV_ERR_INVALID, "fv_device_count: null output");
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess) {
    *out_count = 0;
    return fv_fail(FV_ERR_HIP, "hipGetDeviceCount failed: %s", hipGetErrorString(e));
  }
  *out_count = n;
  return FV_OK;
}

extern "C" int fv_set_device(int device) {
  FV_HIP(hipSetDevice(device));
  return FV_OK;
}

extern "C" int fv_device_info(char *name, size_t name_cap, int *out_compute_units,
                              uint64_t *out_hbm_bytes) {
  int dev = 0;
  FV_HIP(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  FV_HIP(hipGetDeviceProperties(&prop, dev));
  if (name && name_cap) {
    snprintf(name, name_cap, "%s (%s)", prop.name, prop.gcnArchName);
  }
  if (out_compute_units) *out_compute_units = prop.multiProcessorCount;
  if (out_hbm_bytes) *out_hbm_bytes = (uint64_t)prop.totalGlobalMem;
  return FV_OK;
}

extern "C" int fv_device_memory(uint64_t *out_free_bytes, uint64_t *out_total_bytes) {
  size_t free_b = 0, total_b = 0;
  FV_HIP(hipMemGetInfo(&free_b, &total_b));
  if (out_free_bytes) *out_free_bytes = (uint64_t)free_b;
  if (out_total_bytes) *out_total_bytes = (uint64_t)total_b;
  return FV_OK;
}

extern "C" int fv_host_alloc_pinned(size_t bytes, void **out_ptr) {
  FV_REQUIRE(out_ptr, FV_ERR_INVALID, "fv_host_alloc_pinned: null output");
  *out_ptr = nullptr;
  if (bytes == 0) return FV_OK;
  FV_HIP(hipHostMalloc(out_ptr, bytes, hipHostMallocDefault));
  return FV_OK;
}

extern "C" int fv_host_free_pinned(void *ptr) {
  if (ptr) FV_HIP(hipHostFree(ptr));
  return FV_OK;
}

extern "C" int fv_dev_alloc(size_t bytes, void **out_dev_ptr) {
  FV_REQUIRE(out_dev_ptr, FV_ERR_INVALID, "fv_dev_alloc: null output");
  *out_dev_ptr = nullptr;
  if (bytes == 0) return FV_OK;
  FV_HIP(hipMalloc(out_dev_ptr, bytes));
  return FV_OK;
}

extern "C" int fv_dev_free(void *dev_ptr) {
  if (dev_ptr) FV_HIP(hipFree(dev_ptr));
  return FV_OK;
}

extern "C" int fv_dev_upload(void *dst_dev, const void *src_host, size_t bytes) {
  if (bytes == 0) return FV_OK;
  FV_REQUIRE(dst_dev && src_host, FV_ERR_INVALID, "fv_dev_upload: null pointer");
  FV_HIP(hipMemcpy(dst_dev, src_host, bytes, hipMemcpyHostToDevice));
  return FV_OK;
}

extern "C" int fv_dev_download(void *dst_host, const void *src_dev, size_t bytes) {
  if (bytes == 0) return FV_OK;
  FV_REQUIRE(dst_host && src_dev, FV_ERR_INVALID, "fv_dev_download: null pointer");
  FV_HIP(hipMemcpy(dst_host, src_dev, bytes, hipMemcpyDeviceToHost));
  return FV_OK;
}

// ---- layout change ------------------------------------------------------------------
// 64 x 64 tiles through LDS (+1 padding column against bank conflicts): reads are coalesced
// along N of the row-major matrix, writes along K of the token-major one (and vice versa).

#define FV_TT 64

// W: K x N of a row-major matrix of `pitch` columns; Wt: where its first column's first row goes. Of Wt's rows the
// elements from K up to `last` are written as zeros.
__global__ __launch_bounds__(256) void fv_to_token_major_kernel(const float *__restrict__ W, uint64_t pitch,
                                                                float *__restrict__ Wt, uint32_t K,
                                                                uint64_t N, uint32_t ldk, uint32_t last) {
  __shared__ float tile[FV_TT][FV_TT + 1];
  const uint64_t i0 = (uint64_t)blockIdx.x * FV_TT;  // token (column of W)
  const uint32_t h0 = blockIdx.y * FV_TT;            // neuron (row of W)
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < FV_TT; r += 4) {
    uint32_t h = h0 + r;
    uint64_t i = i0 + tx;
    tile[r][tx] = (h < K && i < N) ? W[(uint64_t)h * pitch + i] : 0.0f;
  }
  __syncthreads();
  for (int r = ty; r < FV_TT; r += 4) {
    uint64_t i = i0 + r;
    uint32_t h = h0 + tx;
    if (i < N && h < last) Wt[i * ldk + h] = tile[tx][r];
  }
}

__global__ __launch_bounds__(256) void fv_to_row_major_kernel(const float *__restrict__ Wt,
                                                              float *__restrict__ W, uint64_t pitch, uint32_t K,
                                                              uint64_t N, uint32_t ldk) {
  __shared__ float tile[FV_TT][FV_TT + 1];
  const uint64_t i0 = (uint64_t)blockIdx.x * FV_TT;
  const uint32_t h0 = blockIdx.y * FV_TT;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < FV_TT; r += 4) {
    uint64_t i = i0 + r;
    uint32_t h = h0 + tx;
    tile[r][tx] = (i < N && h < K) ? Wt[i * ldk + h] : 0.0f;
  }
  __syncthreads();
  for (int r = ty; r < FV_TT; r += 4) {
    uint32_t h = h0 + r;
    uint64_t i = i0 + tx;
    if (h < K && i < N) W[(uint64_t)h * pitch + i] = tile[tx][r];
  }
}

static int fv_launch_to_token_major(const float *W, uint64_t pitch, float *Wt, uint32_t K, uint64_t N, uint32_t ldk,
                                    uint32_t last, hipStream_t stream) {
  dim3 grid((unsigned)((N + FV_TT - 1) / FV_TT), (last + FV_TT - 1) / FV_TT);
  hipLaunchKernelGGL(fv_to_token_major_kernel, grid, dim3(256), 0, stream, W, pitch, Wt, K, N, ldk, last);
  FV_HIP(hipGetLastError());
  return FV_OK;
}

static int fv_launch_to_row_major(const float *Wt, float *W, uint64_t pitch, uint32_t K, uint64_t N, uint32_t ldk,
                                  hipStream_t stream) {
  dim3 grid((unsigned)((N + FV_TT - 1) / FV_TT), (K + FV_TT - 1) / FV_TT);
  hipLaunchKernelGGL(fv_to_row_major_kernel, grid, dim3(256), 0, stream, Wt, W, pitch, K, N, ldk);
  FV_HIP(hipGetLastError());
  return FV_OK;
}

// ---- transfers to and from host memory -----------------------------------------------------------------------

// The device's address of `bytes` of page-locked host memory at p (hipHostMalloc), or null where the range is anything
// else: pageable, or not inside one allocation.
static void *fv_device_view(const void *p, size_t bytes) {
  hipPointerAttribute_t at;
  void *base = nullptr;
  size_t size = 0;
  if (hipPointerGetAttributes(&at, p) != hipSuccess || at.type != hipMemoryTypeHost || !at.devicePointer ||
      hipMemGetAddressRange((hipDeviceptr_t *)&base, &size, (hipDeviceptr_t)at.devicePointer) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  const size_t before = (size_t)((char *)at.devicePointer - (char *)base);
  return before <= size && bytes <= size - before ? at.devicePointer : nullptr;
}

bool fv_is_pageable(const void *p) {
  hipPointerAttribute_t at;
  if (hipPointerGetAttributes(&at, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return at.type == hipMemoryTypeUnregistered;
}

// The process's page-locked slots: made when first needed, up to fv_stage_most, kept for the transfers that follow
// (page-locking 4 MB takes 0.1 to 0.8 ms) until fv_host_staging_release.
static std::mutex fv_stage_mutex;
static std::condition_variable fv_stage_returned;
static char *fv_stage_idle[FV_STAGE_SLOTS_MAX];
static unsigned fv_stage_n_idle = 0, fv_stage_made = 0, fv_stage_most = FV_STAGE_SLOTS_MAX;

// (with the lock held)
static void fv_stage_trim(unsigned keep) {
  while (fv_stage_n_idle && fv_stage_made > keep) {
    (void)hipHostFree(fv_stage_idle[--fv_stage_n_idle]);
    fv_stage_made--;
  }
}

fv_stage_lease::fv_stage_lease(unsigned want) {
  std::unique_lock<std::mutex> lock(fv_stage_mutex);
  while (n < want && n < FV_STAGE_SLOTS_LEASED) {
    char *p = nullptr;
    if (fv_stage_n_idle) {
      p = fv_stage_idle[--fv_stage_n_idle];
    } else if (fv_stage_made < fv_stage_most) {
      if (hipHostMalloc((void **)&p, FV_STAGE_SLOT_BYTES, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        break;  // with fewer than wanted, or none
      }
      fv_stage_made++;
    } else if (n == 0 && fv_stage_made) {
      fv_stage_returned.wait(lock);
      continue;
    } else {
      break;
    }
    if (hipEventCreateWithFlags(&events[n], hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      fv_stage_idle[fv_stage_n_idle++] = p;
      fv_stage_returned.notify_all();
      break;
    }
    slots[n++] = p;
  }
}

fv_stage_lease::~fv_stage_lease() {
  for (unsigned i = 0; i < n; ++i) (void)hipEventDestroy(events[i]);
  {
    std::lock_guard<std::mutex> lock(fv_stage_mutex);
    for (unsigned i = 0; i < n; ++i) fv_stage_idle[fv_stage_n_idle++] = slots[i];
    fv_stage_trim(fv_stage_most);
  }
  fv_stage_returned.notify_all();
}

// Idle streams, each with its device; as many are made as calls have held at once, and kept until
// fv_host_staging_release.
struct fv_idle_stream {
  int device;
  hipStream_t stream;
};
static std::vector<fv_idle_stream> fv_streams_idle;

int fv_stream_lease::take(bool make) {
  FV_HIP(hipGetDevice(&device));
  {
    std::lock_guard<std::mutex> lock(fv_stage_mutex);
    for (size_t i = 0; i < fv_streams_idle.size(); ++i)
      if (fv_streams_idle[i].device == device) {
        stream = fv_streams_idle[i].stream;
        fv_streams_idle.erase(fv_streams_idle.begin() + (ptrdiff_t)i);
        return FV_OK;
      }
  }
  if (make) FV_HIP(hipStreamCreate(&stream));
  return FV_OK;
}

fv_stream_lease::~fv_stream_lease() {
  if (!stream) return;
  std::lock_guard<std::mutex> lock(fv_stage_mutex);
  if (fv_streams_idle.size() < FV_STAGE_SLOTS_MAX)
    fv_streams_idle.push_back({device, stream});
  else
    (void)hipStreamDestroy(stream);
}

extern "C" int fv_host_staging_held(size_t *out_bytes) {
  FV_REQUIRE(out_bytes, FV_ERR_INVALID, "null argument");
  std::lock_guard<std::mutex> lock(fv_stage_mutex);
  *out_bytes = fv_stage_made * FV_STAGE_SLOT_BYTES;
  return FV_OK;
}

extern "C" int fv_host_staging_limit(size_t bytes) {
  std::lock_guard<std::mutex> lock(fv_stage_mutex);
  const size_t slots = bytes / FV_STAGE_SLOT_BYTES;
  fv_stage_most = slots < FV_STAGE_SLOTS_MAX ? (unsigned)slots : FV_STAGE_SLOTS_MAX;
  fv_stage_trim(fv_stage_most);
  fv_stage_returned.notify_all();
  return FV_OK;
}

extern "C" int fv_host_staging_release(void) {
  std::lock_guard<std::mutex> lock(fv_stage_mutex);
  fv_stage_trim(0);
  for (const fv_idle_stream &idle : fv_streams_idle) (void)hipStreamDestroy(idle.stream);
  fv_streams_idle.clear();
  return FV_OK;
}

// Both ends: the range may begin or end inside page-locked memory of the caller's.
static bool fv_pageable_range(const void *host, size_t bytes) {
  return fv_is_pageable(host) && fv_is_pageable((const char *)host + bytes - 1);
}

int fv_copy_up(void *dst_dev, const void *src_host, size_t bytes, hipStream_t stream) {
  if (bytes == 0) return FV_OK;
  fv_stage_lease lease(fv_upload_staged(bytes) && fv_pageable_range(src_host, bytes) ? fv_copy_slots(bytes) : 0);
  if (!lease.n) {
    FV_HIP(hipMemcpyAsync(dst_dev, src_host, bytes, hipMemcpyHostToDevice, stream));
    return FV_OK;
  }
  return fv_pipe_up(
      lease, fv_copy_pieces(bytes), stream,
      [&](uint64_t t, char *p) {
        return fv_copy_ring::item{(const char *)src_host + t * FV_STAGE_SLOT_BYTES, p, fv_copy_piece_bytes(bytes, t), 0, 0, 1};
      },
      [&](uint64_t t, char *p) -> int {
        FV_HIP(hipMemcpyAsync((char *)dst_dev + t * FV_STAGE_SLOT_BYTES, p, fv_copy_piece_bytes(bytes, t),
                              hipMemcpyHostToDevice, stream));
        return FV_OK;
      });
}

int fv_copy_down(void *dst_host, const void *src_dev, size_t bytes, hipStream_t stream) {
  if (bytes == 0) return FV_OK;
  fv_stage_lease lease(fv_download_staged(bytes) && fv_pageable_range(dst_host, bytes) ? fv_copy_slots(bytes) : 0);
  if (!lease.n) {
    FV_HIP(hipMemcpyAsync(dst_host, src_dev, bytes, hipMemcpyDeviceToHost, stream));
    FV_HIP(hipStreamSynchronize(stream));
    return FV_OK;
  }
  return fv_pipe_down(
      lease, fv_copy_pieces(bytes), stream,
      [&](uint64_t t, char *p) -> int {
        FV_HIP(hipMemcpyAsync(p, (const char *)src_dev + t * FV_STAGE_SLOT_BYTES, fv_copy_piece_bytes(bytes, t),
                              hipMemcpyDeviceToHost, stream));
        return FV_OK;
      },
      [&](uint64_t t, char *p) {
        return fv_copy_ring::item{p, (char *)dst_host + t * FV_STAGE_SLOT_BYTES, fv_copy_piece_bytes(bytes, t), 0, 0, 1};
      });
}

// One piece of a matrix between the caller's memory (rows of N floats) and a slot (rows of m.pitch floats). Row by row
// also where the rows touch: one memcpy of 4 MB goes past the caches (232 us for an upload, 195 by rows).
static fv_copy_ring::item fv_matrix_item(const fv_matrix_piece &m, uint64_t N, const float *from, float *to, bool up) {
  const size_t row = m.cols * sizeof(float), caller = N * sizeof(float), slot = m.pitch * sizeof(float);
  return {(const char *)from, (char *)to, row, up ? caller : slot, up ? slot : caller, m.rows};
}

static int fv_finish_matrix(int rc, hipStream_t stream, const char *what) {
  const hipError_t e = hipStreamSynchronize(stream);
  if (rc == FV_OK && e != hipSuccess) rc = fv_fail(FV_ERR_HIP, "weight %s failed: %s", what, hipGetErrorString(e));
  return rc;
}

// Page-locked matrices are read and written in place by the layout change, and pageable ones of the sizes that
// fv_host_plan.h names through page-locked slots: there is no staging matrix on the device, whose allocation and release
// (which waits for the device) cost more than the copy of a small matrix, and no second pass over it. The others, and
// memory of any other kind, take the runtime's copies.
int fv_upload_weights(const float *W_host, float *Wt_dev, uint32_t K, uint64_t N, uint32_t ldk,
                      hipStream_t stream) {
  const size_t bytes = (size_t)K * N * sizeof(float);
  int rc = FV_OK;
  if (const float *view = (const float *)fv_device_view(W_host, bytes)) {
    rc = fv_launch_to_token_major(view, N, Wt_dev, K, N, ldk, ldk, stream);
    return fv_finish_matrix(rc, stream, "upload");
  }
  const fv_matrix_pieces pieces = fv_cut_matrix(K, N);
  fv_stage_lease lease(fv_matrix_upload_staged(bytes) && fv_pageable_range(W_host, bytes) ? fv_matrix_slots(&pieces) : 0);
  if (lease.n) {
    return fv_pipe_up(
        lease, pieces.n, stream,
        [&](uint64_t t, char *p) {
          const fv_matrix_piece m = fv_matrix_piece_at(&pieces, t);
          return fv_matrix_item(m, N, W_host + m.h * N + m.i, (float *)p, true);
        },
        [&](uint64_t t, char *p) {
          const fv_matrix_piece m = fv_matrix_piece_at(&pieces, t);
          return fv_launch_to_token_major((const float *)p, m.pitch, Wt_dev + m.i * ldk + m.h, m.rows, m.cols, ldk,
                                          m.h + m.rows == K ? ldk - m.h : m.rows, stream);
        });
  }
  float *on_device = nullptr;
  FV_HIP(hipMalloc((void **)&on_device, bytes));
  const hipError_t e = hipMemcpyAsync(on_device, W_host, bytes, hipMemcpyHostToDevice, stream);
  if (e != hipSuccess) rc = fv_fail(FV_ERR_HIP, "weight upload failed: %s", hipGetErrorString(e));
  if (rc == FV_OK) rc = fv_launch_to_token_major(on_device, N, Wt_dev, K, N, ldk, ldk, stream);
  rc = fv_finish_matrix(rc, stream, "upload");
  (void)hipFree(on_device);
  return rc;
}

int fv_download_weights(const float *Wt_dev, float *W_host, uint32_t K, uint64_t N, uint32_t ldk,
                        hipStream_t stream) {
  const size_t bytes = (size_t)K * N * sizeof(float);
  int rc = FV_OK;
  if (float *view = (float *)fv_device_view(W_host, bytes)) {
    rc = fv_launch_to_row_major(Wt_dev, view, N, K, N, ldk, stream);
    return fv_finish_matrix(rc, stream, "download");
  }
  const fv_matrix_pieces pieces = fv_cut_matrix(K, N);
  fv_stage_lease lease(fv_pageable_range(W_host, bytes) ? fv_matrix_slots(&pieces) : 0);
  if (lease.n) {
    return fv_pipe_down(
        lease, pieces.n, stream,
        [&](uint64_t t, char *p) {
          const fv_matrix_piece m = fv_matrix_piece_at(&pieces, t);
          return fv_launch_to_row_major(Wt_dev + m.i * ldk + m.h, (float *)p, m.pitch, m.rows, m.cols, ldk, stream);
        },
        [&](uint64_t t, char *p) {
          const fv_matrix_piece m = fv_matrix_piece_at(&pieces, t);
          return fv_matrix_item(m, N, (const float *)p, W_host + m.h * N + m.i, false);
        });
  }
  float *on_device = nullptr;
  FV_HIP(hipMalloc((void **)&on_device, bytes));
  rc = fv_launch_to_row_major(Wt_dev, on_device, N, K, N, ldk, stream);
  if (rc == FV_OK) {
    const hipError_t e = hipMemcpyAsync(W_host, on_device, bytes, hipMemcpyDeviceToHost, stream);
    if (e != hipSuccess) rc = fv_fail(FV_ERR_HIP, "weight download failed: %s", hipGetErrorString(e));
  }
  rc = fv_finish_matrix(rc, stream, "download");
  (void)hipFree(on_device);
  return rc;
}

// ---- calibration copy -------------------------------------------------------------------------------
// A plain streaming copy of known size: the yardstick hardware byte counters are scaled by, and a
// measured ceiling for this machine's copy bandwidth.

__global__ __launch_bounds__(256) void fv_calibration_copy_kernel(const float4 *__restrict__ src,
                                                                  float4 *__restrict__ dst, uint64_t n4) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (uint64_t)gridDim.x * 256)
    dst[i] = src[i];
}

extern "C" int fv_calibration_copy(size_t bytes, uint32_t reps, float *out_mean_ms) {
  FV_REQUIRE(bytes >= 16 && reps >= 1 && out_mean_ms, FV_ERR_INVALID, "fv_calibration_copy: bad arguments");
  const uint64_t n4 = bytes / 16;
  float4 *src = nullptr, *dst = nullptr;
  FV_HIP(hipMalloc((void **)&src, n4 * 16));
  hipError_t e = hipMalloc((void **)&dst, n4 * 16);
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (e == hipSuccess) e = hipMemset(src, 1, n4 * 16);
  if (e == hipSuccess) e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  if (e == hipSuccess) {
    const unsigned blocks = 256 * 8;
    hipLaunchKernelGGL(fv_calibration_copy_kernel, dim3(blocks), dim3(256), 0, 0, src, dst, n4);  // warm-up
    e = hipEventRecord(e0, 0);
    for (uint32_t r = 0; r < reps; ++r)
      hipLaunchKernelGGL(fv_calibration_copy_kernel, dim3(blocks), dim3(256), 0, 0, src, dst, n4);
    if (e == hipSuccess) e = hipEventRecord(e1, 0);
    if (e == hipSuccess) e = hipEventSynchronize(e1);
    float ms = 0.0f;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
    *out_mean_ms = ms / (float)reps;
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  (void)hipFree(src);
  (void)hipFree(dst);
  if (e != hipSuccess) return fv_fail(FV_ERR_HIP, "calibration copy failed: %s", hipGetErrorString(e));
  return FV_OK;
}
