// Shared host-side plumbing for the fdk_amd library: error state, status
// macros and small device-memory RAII.  No reference counterpart beyond the
// reference's VERIFY_TRUE / CUDA_CHECK_ERROR (common/type.h:194-196,
// common/cudaLib.cuh:49-56), which throw; this library returns status codes.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstddef>
#include <cstdint>

#include "fdk_amd.h"

namespace fdk {

// Word 3 of a buffer resource for raw (untyped) dword access on gfx9 / CDNA:
// data format 32, no swizzle.  Loads past the resource's byte size return 0.
constexpr int kRawRsrcWord3 = 0x00020000;

// Records a printf-style message as the calling thread's last error and
// returns code, so call sites can `return fail(...)`.
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

// Stream-ordered allocation from the library's per-device staging pool
// (release with hipFreeAsync on a stream).  Freed blocks stay mapped in the
// pool until the process ends, so a batch-sized staging buffer is mapped once,
// not on every call.
int stage_alloc(void** p, size_t bytes, hipStream_t st);

// Device memory a call needs only while its kernels run, on the stream's device.
// scratch_get takes it from blocks kept per device, at most kScratchKeep bytes of them in
// use and idle, and scratch_put gives it back behind the work queued on `st`: the next
// user's stream waits for that work, so blocks pass between streams and threads.  Neither
// waits on the host; but a request larger than every idle block frees those whose work is
// done where that makes room, and hipFree waits for the device: once as sizes grow.
// Requests past the limit are stream-ordered allocations, gone when the call's work is.
// Not for streams being captured.  scratch_get returns FDK_ERR_OOM without a last-error
// message: the caller does without.  scratch_trim frees the current device's idle blocks.
struct ScratchBlock {
  void* p = nullptr;
  size_t bytes = 0;
  hipEvent_t done = nullptr;  // behind the last user's work
  ScratchBlock* next = nullptr;
  int device = 0;
  bool ready = false;
};
struct Scratch {
  void* p = nullptr;
  ScratchBlock* block = nullptr;  // null: a stream-ordered allocation
};
constexpr size_t kScratchKeep = 512u << 20;
int scratch_get(Scratch* s, size_t bytes, hipStream_t st);
void scratch_put(Scratch* s, hipStream_t st);
void scratch_trim();

// hipMalloc, once more with the idle scratch blocks freed where memory is short.
hipError_t dev_malloc(void** p, size_t bytes);

}  // namespace fdk

#define FDK_HIP(call)                                                                  \
  do {                                                                                 \
    hipError_t fdk_e_ = (call);                                                        \
    if (fdk_e_ != hipSuccess)                                                          \
      return ::fdk::fail(fdk_e_ == hipErrorOutOfMemory ? FDK_ERR_OOM : FDK_ERR_HIP,    \
                         "%s failed: %s (%s:%d)", #call, hipGetErrorString(fdk_e_),    \
                         __FILE__, __LINE__);                                          \
  } while (0)

#define FDK_REQUIRE(cond, ...)                                \
  do {                                                        \
    if (!(cond)) return ::fdk::fail(FDK_ERR_INVALID, __VA_ARGS__); \
  } while (0)
