// The scratch list of csrc/capi.cpp over a stand-in for the HIP runtime: memory is counted,
// never touched; an event is done when finish() says so; every call that waits on the host
// is counted.  Prints the first expectation that does not hold.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <set>
#include <thread>
#include <vector>

#include "common.hpp"

namespace {

std::recursive_mutex mu;
struct Event {
  hipStream_t on = nullptr;
  bool recorded = false, done = true;
};
std::map<void*, std::pair<size_t, int>> blocks;  // hipMalloc: bytes, device
std::set<void*> ordered;                         // hipMallocAsync
std::set<Event*> events;
int waits = 0, frees = 0, device = 0;
size_t room = ~(size_t)0;
uintptr_t next_ptr = 0x1000;
std::vector<std::pair<hipStream_t, Event*>> stream_waits;

// streams of device d: 16 d + 1 ..
hipStream_t stream(int n, int d = 0) { return reinterpret_cast<hipStream_t>((uintptr_t)(16 * d + n)); }
int device_of(hipStream_t s) { return (int)((uintptr_t)s / 16); }
size_t held() {
  size_t n = 0;
  for (auto& b : blocks) n += b.second.first;
  return n;
}
void finish() {
  for (Event* e : events) e->done = true;
}
void* fresh() { return reinterpret_cast<void*>(next_ptr += 0x1000); }
Event* ev(hipEvent_t e) { return reinterpret_cast<Event*>(e); }

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::recursive_mutex> l(mu);
  if (held() + n > room) return hipErrorOutOfMemory;
  *p = fresh();
  blocks[*p] = {n, device};
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::recursive_mutex> l(mu);
  ++frees;
  return blocks.erase(p) ? hipSuccess : hipErrorInvalidValue;
}
hipError_t hipMallocAsync(void** p, size_t, hipStream_t) {
  std::lock_guard<std::recursive_mutex> l(mu);
  *p = fresh();
  ordered.insert(*p);
  return hipSuccess;
}
hipError_t hipFreeAsync(void* p, hipStream_t) {
  std::lock_guard<std::recursive_mutex> l(mu);
  return ordered.erase(p) ? hipSuccess : hipErrorInvalidValue;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  std::lock_guard<std::recursive_mutex> l(mu);
  Event* n = new Event;
  events.insert(n);
  *e = reinterpret_cast<hipEvent_t>(n);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  std::lock_guard<std::recursive_mutex> l(mu);
  events.erase(ev(e));
  delete ev(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::recursive_mutex> l(mu);
  ev(e)->on = s;
  ev(e)->recorded = true;
  ev(e)->done = false;
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) { return ev(e)->done ? hipSuccess : hipErrorNotReady; }
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::recursive_mutex> l(mu);
  if (!ev(e)->done) ++waits;
  ev(e)->done = true;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  std::lock_guard<std::recursive_mutex> l(mu);
  stream_waits.push_back({s, ev(e)});
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  ++waits;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = device;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  device = d;
  return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) {
  *d = s ? device_of(s) : device;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetDeviceCount(int* n) {
  *n = 2;
  return hipSuccess;
}
// not reached
hipError_t hipMemPoolCreate(hipMemPool_t*, const hipMemPoolProps*) { return hipErrorInvalidValue; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { return hipErrorInvalidValue; }
hipError_t hipMemPoolDestroy(hipMemPool_t) { return hipErrorInvalidValue; }
hipError_t hipMallocFromPoolAsync(void**, size_t, hipMemPool_t, hipStream_t) { return hipErrorInvalidValue; }
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipErrorInvalidValue; }
hipError_t hipMemcpy2D(void*, size_t, const void*, size_t, size_t, size_t, hipMemcpyKind) { return hipErrorInvalidValue; }
hipError_t hipMemset(void*, int, size_t) { return hipErrorInvalidValue; }
}

#define EXPECT(c)                                     \
  do {                                                \
    if (!(c)) {                                       \
      std::printf("line %d: %s\n", __LINE__, #c);     \
      std::exit(1);                                   \
    }                                                 \
  } while (0)

int main(int argc, char** argv) {
  using fdk::Scratch;
  const size_t MiB = 1u << 20;
  const std::string which = argc > 1 ? argv[1] : "";
  Scratch a, b, c;
  if (which == "hand-over") {
    EXPECT(fdk::scratch_get(&a, 100 * MiB, stream(1)) == FDK_OK && a.p);
    void* p = a.p;
    fdk::scratch_put(&a, stream(1));
    EXPECT(fdk::scratch_get(&b, 80 * MiB, stream(2)) == FDK_OK && b.p == p);
    EXPECT(stream_waits.size() == 1 && stream_waits[0].first == stream(2));  // behind stream 1's work
    EXPECT(stream_waits[0].second->on == stream(1) && waits == 0);
    EXPECT(fdk::scratch_get(&c, 80 * MiB, stream(1)) == FDK_OK && c.p != p);  // not while b has it
    fdk::scratch_put(&b, stream(2));
    fdk::scratch_put(&c, stream(1));
  } else if (which == "two streams past the limit") {
    for (int turn = 0; turn < 4; ++turn) {
      EXPECT(fdk::scratch_get(&a, 258 * MiB, stream(1)) == FDK_OK && a.p);
      EXPECT(fdk::scratch_get(&b, 258 * MiB, stream(2)) == FDK_OK && b.p && b.p != a.p);
      fdk::scratch_put(&a, stream(1));
      fdk::scratch_put(&b, stream(2));
      EXPECT(waits == 0 && frees == 0 && held() <= fdk::kScratchKeep);
    }
    EXPECT(ordered.empty());
  } else if (which == "larger while busy") {
    EXPECT(fdk::scratch_get(&a, 300 * MiB, stream(1)) == FDK_OK);
    fdk::scratch_put(&a, stream(1));
    EXPECT(fdk::scratch_get(&b, 400 * MiB, stream(2)) == FDK_OK && b.p);  // stream 1 is not waited for
    EXPECT(waits == 0 && frees == 0);
    fdk::scratch_put(&b, stream(2));
    finish();
    EXPECT(fdk::scratch_get(&b, 400 * MiB, stream(2)) == FDK_OK && b.p);  // its block makes room now
    EXPECT(waits == 0 && frees == 1 && blocks.count(b.p) && held() <= fdk::kScratchKeep);
    fdk::scratch_put(&b, stream(2));
  } else if (which == "larger beside a smaller") {
    // an idle block goes only where that makes room
    EXPECT(fdk::scratch_get(&a, 400 * MiB, stream(1)) == FDK_OK);
    EXPECT(fdk::scratch_get(&b, 100 * MiB, stream(2)) == FDK_OK);
    fdk::scratch_put(&b, stream(2));
    finish();
    EXPECT(fdk::scratch_get(&c, 200 * MiB, stream(2)) == FDK_OK && c.p && frees == 0);
    fdk::scratch_put(&c, stream(2));
    fdk::scratch_put(&a, stream(1));
    EXPECT(held() <= fdk::kScratchKeep);
  } else if (which == "other device") {
    EXPECT(fdk::scratch_get(&a, 10 * MiB, stream(1, 1)) == FDK_OK && a.p);
    EXPECT(blocks[a.p].second == 1 && device == 0);  // beside the stream, not on the current device
    void* p = a.p;
    fdk::scratch_put(&a, stream(1, 1));
    EXPECT(fdk::scratch_get(&b, 10 * MiB, stream(1)) == FDK_OK && b.p != p && blocks[b.p].second == 0);
    fdk::scratch_put(&b, stream(1));
    EXPECT(fdk::scratch_get(&a, 10 * MiB, stream(2, 1)) == FDK_OK && a.p == p && device == 0);
    fdk::scratch_put(&a, stream(2, 1));
  } else if (which == "out of memory") {
    room = 150 * MiB;
    EXPECT(fdk::scratch_get(&a, 100 * MiB, stream(1)) == FDK_OK);
    EXPECT(fdk::scratch_get(&b, 100 * MiB, stream(1)) == FDK_ERR_OOM && !b.p);
    fdk::scratch_put(&a, stream(1));
    fdk::scratch_trim();
    EXPECT(held() == 0);
    for (int turn = 0; turn < 3; ++turn) {  // the refused requests do not count against the limit
      EXPECT(fdk::scratch_get(&b, 140 * MiB, stream(1)) == FDK_OK && blocks.count(b.p));
      EXPECT(fdk::scratch_get(&a, 140 * MiB, stream(1)) == FDK_ERR_OOM);
      fdk::scratch_put(&b, stream(1));
    }
    void* p = nullptr;
    EXPECT(fdk_dev_malloc(&p, 120 * MiB) == FDK_OK && p && held() == 120 * MiB);  // the kept block made room
  } else if (which == "threads") {
    std::atomic<bool> twice{false};
    std::mutex own_mu;
    std::set<void*> own;
    std::vector<std::thread> t;
    for (int n = 1; n <= 8; ++n)
      t.emplace_back([&, n] {
        for (int k = 0; k < 500; ++k) {
          Scratch s;
          if (fdk::scratch_get(&s, (size_t)((k * n) % 90 + 1) * MiB, stream(n)) != FDK_OK) continue;
          {
            std::lock_guard<std::mutex> l(own_mu);
            if (!own.insert(s.p).second) twice = true;
          }
          std::this_thread::yield();
          {
            std::lock_guard<std::mutex> l(own_mu);
            own.erase(s.p);
          }
          fdk::scratch_put(&s, stream(n));
        }
      });
    for (auto& q : t) q.join();
    EXPECT(!twice && held() <= fdk::kScratchKeep && ordered.empty());
    finish();
    fdk::scratch_trim();
    EXPECT(held() == 0 && events.empty());
  } else {
    EXPECT(!"unknown check");
  }
  return 0;
}
