// The few runtime calls that akx_copy.hpp makes, on the host: a stream is a
// queue whose copies happen when something waits for them, in order, so that a
// staging buffer overwritten too early shows; page-locked memory can run out.
#pragma once

#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

struct FakeStream {
  struct Copy {
    void* to;
    const void* from;
    size_t bytes;
  };
  std::mutex m;
  std::vector<Copy> queue;
  size_t done = 0;
  void wait(size_t upto) {
    std::lock_guard<std::mutex> g(m);
    for (; done < upto; ++done) std::memcpy(queue[done].to, queue[done].from, queue[done].bytes);
  }
};
struct FakeEvent {
  FakeStream* stream = nullptr;
  size_t at = 0;
};
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;

inline std::mutex fake_mutex;
inline long fake_pinned_left = 1 << 20;  // page-locked buffers that may still be had

inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  std::lock_guard<std::mutex> g(fake_mutex);
  if (fake_pinned_left <= 0) return hipErrorOutOfMemory;
  --fake_pinned_left;
  *p = std::malloc(n);
  std::memset(*p, 0xA5, n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipMalloc(void** p, size_t n) {
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind,
                                 hipStream_t s) {
  std::lock_guard<std::mutex> g(s->m);
  s->queue.push_back({to, from, n});
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  size_t upto;
  {
    std::lock_guard<std::mutex> g(s->m);
    upto = s->queue.size();
  }
  s->wait(upto);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new FakeEvent;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::mutex> g(s->m);
  e->stream = s;
  e->at = s->queue.size();
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  if (e->stream) e->stream->wait(e->at);
  return hipSuccess;
}
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
