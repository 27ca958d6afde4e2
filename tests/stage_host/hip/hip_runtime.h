// A host-only stand-in for the HIP calls of genesis6_amd/csrc/g6_stage.h:
// "device" memory is host memory, a stream holds its copies until something
// waits for them (or carries them out at once), events belong to the device
// that was current when they were made, and every copied byte is counted.
#pragma once
#include <stdlib.h>
#include <string.h>

#include <condition_variable>
#include <mutex>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorInvalidHandle, hipErrorOutOfMemory };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
enum hipMemcpyKind { hipMemcpyDeviceToHost };

namespace stub {
inline std::mutex mu;
inline std::condition_variable cv;
inline int device = 0, pinned = 0, events = 0;
inline bool eager = false, out_of_memory = false;
inline size_t bytes = 0;
struct Copy {
  void *dst;
  const void *src;
  size_t len;
};
struct Stream {
  int dev = 0;
  bool busy = false;  // work ahead of the copies that does not end yet
  std::vector<Copy> todo;
  size_t done = 0;
};
struct Event {
  int dev;
  Stream *s = nullptr;
  size_t upto = 0;
};
inline void finish(std::unique_lock<std::mutex> &lk, Stream *s, size_t upto) {
  cv.wait(lk, [&] { return !s->busy; });
  for (; s->done < upto; s->done++)
    memcpy(s->todo[s->done].dst, s->todo[s->done].src, s->todo[s->done].len);
}
}  // namespace stub
typedef stub::Stream *hipStream_t;
typedef stub::Event *hipEvent_t;

inline hipError_t hipGetDevice(int *d) {
  *d = stub::device;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
  stub::device = d;
  return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  std::lock_guard<std::mutex> lk(stub::mu);
  if (stub::out_of_memory) return hipErrorOutOfMemory;
  *p = malloc(n);
  stub::pinned++;
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
  std::lock_guard<std::mutex> lk(stub::mu);
  free(p);
  stub::pinned--;
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  std::lock_guard<std::mutex> lk(stub::mu);
  *e = new stub::Event{stub::device};
  stub::events++;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  std::lock_guard<std::mutex> lk(stub::mu);
  delete e;
  stub::events--;
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *dst, const void *src, size_t len, hipMemcpyKind,
                                 hipStream_t s) {
  std::unique_lock<std::mutex> lk(stub::mu);
  s->todo.push_back({dst, src, len});
  stub::bytes += len;
  if (stub::eager) stub::finish(lk, s, s->todo.size());
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::mutex> lk(stub::mu);
  if (e->dev != s->dev) return hipErrorInvalidHandle;
  e->s = s;
  e->upto = s->todo.size();
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  std::unique_lock<std::mutex> lk(stub::mu);
  if (e->s) stub::finish(lk, e->s, e->upto);
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  std::unique_lock<std::mutex> lk(stub::mu);
  stub::finish(lk, s, s->todo.size());
  return hipSuccess;
}
