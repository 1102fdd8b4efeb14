// Error state and device queries of the C ABI (include/fdk_amd.h).
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <utility>

#include "common.hpp"

namespace {
thread_local std::string g_last_error;
}

namespace fdk {

int fail(int code, const char* fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

int stage_alloc(void** p, size_t bytes, hipStream_t st) {
  static std::mutex mu;
  static std::map<int, hipMemPool_t> pools;
  int dev = 0;
  FDK_HIP(hipGetDevice(&dev));
  hipMemPool_t pool = nullptr;
  {
    std::lock_guard<std::mutex> lock(mu);
    auto it = pools.find(dev);
    if (it != pools.end()) {
      pool = it->second;
    } else {
      hipMemPoolProps props{};
      props.allocType = hipMemAllocationTypePinned;
      props.handleTypes = hipMemHandleTypeNone;
      props.location.type = hipMemLocationTypeDevice;
      props.location.id = dev;
      FDK_HIP(hipMemPoolCreate(&pool, &props));
      uint64_t keep = UINT64_MAX;  // freed blocks stay mapped for the next call
      hipError_t e = hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep);
      if (e != hipSuccess) {
        (void)hipMemPoolDestroy(pool);
        return fail(FDK_ERR_HIP, "staging pool: %s", hipGetErrorString(e));
      }
      pools[dev] = pool;
    }
  }
  hipError_t e = hipMallocFromPoolAsync(p, bytes, pool, st);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    scratch_trim();
    e = hipMallocFromPoolAsync(p, bytes, pool, st);
  }
  FDK_HIP(e);
  return FDK_OK;
}

namespace {

// Allocating and freeing would be refused while another thread captures a stream
// in the default mode; these allocations are no part of any graph.
struct Relaxed {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// The device that memory and events are made on, the caller's afterwards.
struct OnDevice {
  int before = -1;
  explicit OnDevice(int dev) {
    int now = dev;
    if (hipGetDevice(&now) == hipSuccess && now != dev && hipSetDevice(dev) == hipSuccess) before = now;
  }
  ~OnDevice() {
    if (before >= 0) (void)hipSetDevice(before);
  }
};

// A device's blocks: those not in use, and the bytes of all of them.
struct ScratchList {
  ScratchBlock* idle = nullptr;
  size_t total = 0;
};
constexpr int kScratchDevices = 64;
std::mutex g_scratch_mutex;
ScratchList g_scratch[kScratchDevices];

// Frees blocks no longer on a list, waiting for the work behind them.
void scratch_free(ScratchBlock* b) {
  Relaxed relaxed;
  while (b) {
    ScratchBlock* next = b->next;
    (void)hipEventSynchronize(b->done);
    (void)hipFree(b->p);
    (void)hipEventDestroy(b->done);
    delete b;
    b = next;
  }
  (void)hipGetLastError();
}

// Takes off the list what is needed of the idle blocks whose work is done, smallest
// first, so that `bytes` more fit the limit; nothing if they would not make room.
ScratchBlock* scratch_make_room(ScratchList& l, size_t bytes) {
  size_t done = 0;
  for (ScratchBlock* b = l.idle; b; b = b->next) {
    b->ready = hipEventQuery(b->done) == hipSuccess;
    if (b->ready) done += b->bytes;
  }
  (void)hipGetLastError();
  ScratchBlock* out = nullptr;
  if (l.total - done + bytes > kScratchKeep) return out;
  while (l.total + bytes > kScratchKeep) {
    ScratchBlock** least = nullptr;
    for (ScratchBlock** q = &l.idle; *q; q = &(*q)->next)
      if ((*q)->ready && (!least || (*q)->bytes < (*least)->bytes)) least = q;
    ScratchBlock* b = *least;
    *least = b->next;
    l.total -= b->bytes;
    b->next = out;
    out = b;
  }
  return out;
}

}  // namespace

void scratch_trim() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev >= kScratchDevices) return;
  ScratchBlock* b = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    std::swap(b, g_scratch[dev].idle);
    for (ScratchBlock* q = b; q; q = q->next) g_scratch[dev].total -= q->bytes;
  }
  scratch_free(b);
}

hipError_t dev_malloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory) return e;
  (void)hipGetLastError();
  scratch_trim();
  return hipMalloc(p, bytes);
}

int scratch_get(Scratch* s, size_t bytes, hipStream_t st) {
  *s = Scratch{};
  int dev = 0;
  if (hipStreamGetDevice(st, &dev) != hipSuccess || dev >= kScratchDevices) {
    (void)hipGetLastError();
    return FDK_ERR_OOM;
  }
  OnDevice here(dev);
  const size_t size = (bytes + (2u << 20) - 1) >> 21 << 21;
  ScratchBlock *b = nullptr, *old = nullptr;
  bool make = false;
  if (size <= kScratchKeep) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    ScratchList& l = g_scratch[dev];
    ScratchBlock** best = nullptr;
    for (ScratchBlock** q = &l.idle; *q; q = &(*q)->next)
      if ((*q)->bytes >= bytes && (!best || (*q)->bytes < (*best)->bytes)) best = q;
    if (best) {
      b = *best;
      *best = b->next;
    } else {
      if (l.total + size > kScratchKeep) old = scratch_make_room(l, size);
      make = l.total + size <= kScratchKeep;
      if (make) l.total += size;
    }
  }
  if (b) {
    if (hipStreamWaitEvent(st, b->done, 0) == hipSuccess) {
      s->p = b->p;
      s->block = b;
      return FDK_OK;
    }
    (void)hipGetLastError();
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    b->next = g_scratch[dev].idle;
    g_scratch[dev].idle = b;
    return FDK_ERR_OOM;
  }
  scratch_free(old);
  if (make) {
    Relaxed relaxed;
    b = new (std::nothrow) ScratchBlock;
    if (b && hipEventCreateWithFlags(&b->done, hipEventDisableTiming) == hipSuccess) {
      if (hipMalloc(&b->p, size) == hipSuccess) {
        b->bytes = size;
        b->device = dev;
        s->p = b->p;
        s->block = b;
        return FDK_OK;
      }
      (void)hipEventDestroy(b->done);
    }
    (void)hipGetLastError();
    delete b;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    g_scratch[dev].total -= size;
    return FDK_ERR_OOM;
  }
  if (hipMallocAsync(&s->p, bytes, st) == hipSuccess) return FDK_OK;
  (void)hipGetLastError();
  *s = Scratch{};
  return FDK_ERR_OOM;
}

void scratch_put(Scratch* s, hipStream_t st) {
  ScratchBlock* b = s->block;
  if (s->p && !b) (void)hipFreeAsync(s->p, st);
  *s = Scratch{};
  if (!b) return;
  const bool behind = hipEventRecord(b->done, st) == hipSuccess;
  if (!behind) (void)hipStreamSynchronize(st);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  b->next = g_scratch[b->device].idle;
  g_scratch[b->device].idle = b;
}

}  // namespace fdk

extern "C" int fdk_last_error(char* buf, size_t len) {
  if (buf && len) {
    std::strncpy(buf, g_last_error.c_str(), len - 1);
    buf[len - 1] = 0;
  }
  return (int)g_last_error.size();
}

extern "C" int fdk_release_scratch(void) {
  fdk::scratch_trim();
  return FDK_OK;
}

extern "C" int fdk_version(void) { return 100; }

extern "C" int fdk_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

// Device buffers for the C++ layer's DevData / DevArray3D (cudaBP/cudaLib.cuh:298-420,
// 552-640): linear allocations on the current device, copies in either direction.
extern "C" int fdk_dev_malloc(void** out, size_t bytes) {
  FDK_REQUIRE(out, "null output pointer");
  *out = nullptr;
  if (bytes == 0) return FDK_OK;
  FDK_HIP(fdk::dev_malloc(out, bytes));
  return FDK_OK;
}

extern "C" int fdk_dev_free(void* p) {
  if (p) FDK_HIP(hipFree(p));
  return FDK_OK;
}

extern "C" int fdk_memcpy(void* dst, const void* src, size_t bytes) {
  if (bytes == 0) return FDK_OK;
  FDK_REQUIRE(dst && src, "null pointer");
  FDK_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDefault));
  return FDK_OK;
}

extern "C" int fdk_memcpy_2d(void* dst, size_t dst_pitch, const void* src, size_t src_pitch,
                             size_t width_bytes, size_t rows) {
  if (width_bytes == 0 || rows == 0) return FDK_OK;
  FDK_REQUIRE(dst && src, "null pointer");
  FDK_REQUIRE(dst_pitch >= width_bytes && src_pitch >= width_bytes, "pitch below row width");
  FDK_HIP(hipMemcpy2D(dst, dst_pitch, src, src_pitch, width_bytes, rows, hipMemcpyDefault));
  return FDK_OK;
}

extern "C" int fdk_dev_memset(void* p, int value, size_t bytes) {
  if (bytes == 0) return FDK_OK;
  FDK_REQUIRE(p, "null pointer");
  FDK_HIP(hipMemset(p, value, bytes));
  return FDK_OK;
}
