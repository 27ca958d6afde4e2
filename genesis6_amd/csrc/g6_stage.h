// Downloads of arrays that lie one after another in device memory: through two
// pinned buffers, the copy of one piece to the host arrays beside the transfer
// of the next.  A copy to pageable memory costs its own staging and
// synchronization per array: the four state arrays took 54 us for 216
// molecules, 113 for 4096 and 1570 for 65,536, and take 25, 86 and 970 in
// pieces of 1 MiB (512 KiB: 26, 102, 1300; 4 MiB: 26, 96, 1030; each piece costs
// about 17 us).
//
// An event may be recorded on the streams of its own device alone, so every
// device has its own buffers and events.  They are made at the device's first
// download and live while a handle on the device does; a download holds them to
// its end, so threads on one device take turns.
#pragma once
#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <mutex>

namespace g6 {

struct HostPart {
  double *p;   // nullptr: skipped
  size_t len;  // doubles
};

constexpr size_t kStageBytes = (size_t)1 << 20;
constexpr int kStageDevices = 64;

struct Staging {
  std::mutex mu;
  int users = 0;
  bool ready = false;
  char *buf[2] = {nullptr, nullptr};
  hipEvent_t ev[2];
};
inline Staging &staging_of(int dev) {
  static Staging all[kStageDevices];
  return all[dev];
}

// a handle on device dev begins and ends
inline void staging_open(int dev) {
  if (dev < 0 || dev >= kStageDevices) return;
  Staging &g = staging_of(dev);
  std::lock_guard<std::mutex> lk(g.mu);
  g.users++;
}
inline void staging_close(int dev) {
  if (dev < 0 || dev >= kStageDevices) return;
  Staging &g = staging_of(dev);
  std::lock_guard<std::mutex> lk(g.mu);
  if (--g.users > 0 || !g.ready) return;
  for (int k = 0; k < 2; k++) {
    (void)hipHostFree(g.buf[k]);
    (void)hipEventDestroy(g.ev[k]);
    g.buf[k] = nullptr;
  }
  g.ready = false;
}

// the buffers and events of device dev (g.mu held)
inline bool staging_make(Staging &g, int dev) {
  if (g.ready) return true;
  int cur = 0;
  if (hipGetDevice(&cur) != hipSuccess) return false;
  if (cur != dev && hipSetDevice(dev) != hipSuccess) return false;
  int nb = 0, ne = 0;
  while (nb < 2 && hipHostMalloc((void **)&g.buf[nb], kStageBytes, hipHostMallocDefault) == hipSuccess) nb++;
  while (nb == 2 && ne < 2 && hipEventCreateWithFlags(&g.ev[ne], hipEventDisableTiming) == hipSuccess) ne++;
  g.ready = nb == 2 && ne == 2;
  if (!g.ready) {
    while (ne > 0) (void)hipEventDestroy(g.ev[--ne]);
    while (nb > 0) (void)hipHostFree(g.buf[--nb]);
    g.buf[0] = g.buf[1] = nullptr;
  }
  if (cur != dev) (void)hipSetDevice(cur);
  return g.ready;
}

// without buffers: each array by itself
inline hipError_t plain_download(hipStream_t stream, const double *src, const HostPart *part,
                                 int np) {
  size_t at = 0;
  for (int k = 0; k < np; k++) {
    if (part[k].p && part[k].len > 0) {
      const hipError_t e = hipMemcpyAsync(part[k].p, src + at, part[k].len * sizeof(double),
                                          hipMemcpyDeviceToHost, stream);
      if (e != hipSuccess) {
        (void)hipStreamSynchronize(stream);
        return e;
      }
    }
    at += part[k].len;
  }
  return hipStreamSynchronize(stream);
}

inline hipError_t staged_download(int dev, hipStream_t stream, const double *src,
                                  const HostPart *part, int np) {
  if (dev < 0 || dev >= kStageDevices) return plain_download(stream, src, part, np);
  Staging &g = staging_of(dev);
  std::lock_guard<std::mutex> lk(g.mu);
  if (!staging_make(g, dev)) {
    (void)hipGetLastError();
    return plain_download(stream, src, part, np);
  }
  size_t total = 0;
  for (int k = 0; k < np; k++) total += part[k].len * sizeof(double);
  const size_t pieces = (total + kStageBytes - 1) / kStageBytes;
  auto piece_len = [&](size_t q) { return std::min(kStageBytes, total - q * kStageBytes); };
  auto issue = [&](size_t q) {
    const hipError_t e = hipMemcpyAsync(g.buf[q & 1], (const char *)src + q * kStageBytes,
                                        piece_len(q), hipMemcpyDeviceToHost, stream);
    return e == hipSuccess ? hipEventRecord(g.ev[q & 1], stream) : e;
  };
  hipError_t rc = pieces > 0 ? issue(0) : hipSuccess;
  for (size_t q = 0; rc == hipSuccess && q < pieces; q++) {
    if (q + 1 < pieces) rc = issue(q + 1);
    if (rc == hipSuccess) rc = hipEventSynchronize(g.ev[q & 1]);
    if (rc != hipSuccess) break;
    size_t at = 0;  // the parts' byte ranges that the piece holds
    const size_t b0 = q * kStageBytes, b1 = b0 + piece_len(q);
    for (int k = 0; k < np; k++) {
      const size_t e = at + part[k].len * sizeof(double);
      const size_t lo = std::max(at, b0), hi = std::min(e, b1);
      if (part[k].p && lo < hi)
        memcpy((char *)part[k].p + (lo - at), g.buf[q & 1] + (lo - b0), hi - lo);
      at = e;
    }
  }
  // no transfer into the buffers is left behind by an error
  if (rc != hipSuccess) (void)hipStreamSynchronize(stream);
  return rc;
}

}  // namespace g6
