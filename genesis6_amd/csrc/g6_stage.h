// Downloads of arrays that lie one after another in device memory: through two
// pinned buffers, the copy of one piece to the host arrays beside the transfer
// of the next.  A copy to pageable memory costs its own staging and
// synchronization per array: the four state arrays took 82 us for 216
// molecules, 106 for 4096 and 1500 for 65,536, and take 18, 76 and 1080 in
// pieces of 1 MiB (pieces of 512 KiB and 4 MiB by the copy engine: 102 and 96 us
// for 4096, 1300 and 1030 for 65,536, where 1 MiB took 79 and 990); the COMs
// alone 15, 14 and 86 before, 13, 17 and 78 now.  Into memory that was not
// touched before, as a fresh array's is, 28 MB take 5.8 ms where a plain copy
// takes 6.3.
// Arrays that the caller skips are not moved.
//
// An event may be recorded on the streams of its own device alone, so every
// device has its own buffers and events.  They are made at the device's first
// download and live while a handle on the device does; a transfer holds them to
// its end, so threads on one device take turns (four threads, 65,536 molecules
// each: 6.5 ms by plain copies, 4.4 in turns).
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
constexpr int kStageParts = 8;  // arrays of one download

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

// send(buffer, src, bytes, stream) queues a transfer into a pinned buffer
template <class Send>
inline hipError_t staged_download(int dev, hipStream_t stream, const double *src,
                                  const HostPart *part, int np, Send &&send) {
  if (dev < 0 || dev >= kStageDevices || np > kStageParts)
    return plain_download(stream, src, part, np);
  // what the stream has queued ends before the buffers are taken, so that a
  // handle at work keeps no other thread from its download
  const hipError_t idle = hipStreamSynchronize(stream);
  if (idle != hipSuccess) return idle;
  Staging &g = staging_of(dev);
  std::lock_guard<std::mutex> lk(g.mu);
  if (!staging_make(g, dev)) {
    (void)hipGetLastError();
    return plain_download(stream, src, part, np);
  }
  // pieces of the wanted arrays' bytes, packed: f(offset in the piece, part,
  // offset in the part, bytes) of each range that bytes [b0, b1) hold
  auto ranges = [&](size_t b0, size_t b1, auto f) {
    size_t at = 0;
    for (int k = 0; k < np; k++) {
      if (!part[k].p) continue;
      const size_t e = at + part[k].len * sizeof(double);
      const size_t lo = std::max(at, b0), hi = std::min(e, b1);
      if (lo < hi) f(lo - b0, k, lo - at, hi - lo);
      at = e;
    }
  };
  size_t total = 0, start[kStageParts], pos = 0;
  for (int k = 0; k < np; k++) {
    if (part[k].p) total += part[k].len * sizeof(double);
    start[k] = pos;
    pos += part[k].len * sizeof(double);
  }
  const size_t pieces = (total + kStageBytes - 1) / kStageBytes;
  auto piece_end = [&](size_t q) { return std::min((q + 1) * kStageBytes, total); };
  auto issue = [&](size_t q) {
    hipError_t e = hipSuccess;
    // neighbouring arrays are one transfer
    size_t from = 0, into = 0, len = 0;
    auto flush = [&] {
      if (len > 0 && e == hipSuccess)
        e = send(g.buf[q & 1] + into, (const char *)src + from, len, stream);
    };
    ranges(q * kStageBytes, piece_end(q), [&](size_t in, int k, size_t off, size_t bytes) {
      if (start[k] + off != from + len) {
        flush();
        from = start[k] + off;
        into = in;
        len = 0;
      }
      len += bytes;
    });
    flush();
    // (a single piece is waited for with the stream: an event costs 7 us)
    if (e == hipSuccess && pieces > 1) e = hipEventRecord(g.ev[q & 1], stream);
    return e;
  };
  hipError_t rc = pieces > 0 ? issue(0) : hipSuccess;
  for (size_t q = 0; rc == hipSuccess && q < pieces; q++) {
    if (q + 1 < pieces) rc = issue(q + 1);
    if (rc == hipSuccess)
      rc = pieces > 1 ? hipEventSynchronize(g.ev[q & 1]) : hipStreamSynchronize(stream);
    if (rc != hipSuccess) break;
    ranges(q * kStageBytes, piece_end(q), [&](size_t in, int k, size_t off, size_t bytes) {
      memcpy((char *)part[k].p + off, g.buf[q & 1] + in, bytes);
    });
  }
  // no transfer into the buffers is left behind by an error
  if (rc != hipSuccess) (void)hipStreamSynchronize(stream);
  return rc;
}

}  // namespace g6
