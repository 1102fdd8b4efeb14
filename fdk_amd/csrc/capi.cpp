// Error state and device queries of the C ABI (include/fdk_amd.h).
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

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
  FDK_HIP(hipMallocFromPoolAsync(p, bytes, pool, st));
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

std::mutex g_scratch_mutex;
std::map<int, std::vector<Scratch>> g_scratch;  // kept blocks, by device

void scratch_free(Scratch& s) {
  Relaxed relaxed;
  (void)hipEventSynchronize(s.done);
  (void)hipFree(s.p);
  (void)hipEventDestroy(s.done);
  (void)hipGetLastError();
  s = Scratch{};
}

// The current device's kept blocks, taken off the list.
std::vector<Scratch> scratch_take_all() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return {};
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  std::vector<Scratch> v;
  v.swap(g_scratch[dev]);
  return v;
}

}  // namespace

void scratch_trim() {
  for (Scratch& s : scratch_take_all()) scratch_free(s);
}

int scratch_get(Scratch* s, size_t bytes, hipStream_t st) {
  *s = Scratch{};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return FDK_ERR_HIP;
  if (bytes > kScratchKeep) {
    s->bytes = bytes;
    if (hipMallocAsync(&s->p, bytes, st) == hipSuccess) return FDK_OK;
    (void)hipGetLastError();
    *s = Scratch{};
    return FDK_ERR_OOM;
  }
  {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    std::vector<Scratch>& v = g_scratch[dev];
    size_t best = v.size();
    for (size_t k = 0; k < v.size(); ++k)
      if (v[k].bytes >= bytes && (best == v.size() || v[k].bytes < v[best].bytes)) best = k;
    if (best < v.size()) {
      *s = v[best];
      v.erase(v.begin() + (long)best);
    }
  }
  if (s->p) {
    if (hipStreamWaitEvent(st, s->done, 0) == hipSuccess) return FDK_OK;
    scratch_free(*s);  // waits for the block's last work instead
  }
  scratch_trim();  // a larger block replaces the kept ones
  Relaxed relaxed;
  s->bytes = (bytes + (2u << 20) - 1) >> 21 << 21;
  if (hipEventCreateWithFlags(&s->done, hipEventDisableTiming) == hipSuccess) {
    if (hipMalloc(&s->p, s->bytes) == hipSuccess) return FDK_OK;
    (void)hipEventDestroy(s->done);
  }
  (void)hipGetLastError();
  *s = Scratch{};
  return FDK_ERR_OOM;
}

void scratch_put(Scratch* s, hipStream_t st) {
  if (!s->p) return;
  if (!s->done) {
    (void)hipFreeAsync(s->p, st);
    *s = Scratch{};
    return;
  }
  int dev = 0;
  if (hipEventRecord(s->done, st) != hipSuccess || hipGetDevice(&dev) != hipSuccess) {
    (void)hipStreamSynchronize(st);
    scratch_free(*s);
    return;
  }
  {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    std::vector<Scratch>& v = g_scratch[dev];
    size_t kept = s->bytes;
    for (const Scratch& q : v) kept += q.bytes;
    if (kept <= kScratchKeep) {
      v.push_back(*s);
      *s = Scratch{};
      return;
    }
  }
  scratch_free(*s);
}

}  // namespace fdk

extern "C" int fdk_last_error(char* buf, size_t len) {
  if (buf && len) {
    std::strncpy(buf, g_last_error.c_str(), len - 1);
    buf[len - 1] = 0;
  }
  return (int)g_last_error.size();
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
  FDK_HIP(hipMalloc(out, bytes));
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
