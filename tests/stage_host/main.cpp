// Checks of genesis6_amd/csrc/g6_stage.h on the host (hip/hip_runtime.h of
// this folder stands in for the runtime).  Each check is an argument; a
// failed one ends the program with status 1.
#include "g6_stage.h"

#include <stdio.h>

#include <chrono>
#include <string>
#include <thread>

using namespace g6;
#define REQUIRE(c)                                          \
  do {                                                      \
    if (!(c)) {                                             \
      printf("line %d: %s does not hold\n", __LINE__, #c);  \
      exit(1);                                              \
    }                                                       \
  } while (0)

// The state arrays of n molecules: a download of the parts in mask; whether
// those come out whole and the others stay untouched.
static bool download(int dev, hipStream_t s, size_t n, int mask) {
  const size_t len[4] = {3 * n, 15 * n, 15 * n, 20 * n};
  std::vector<double> src(53 * n), out[4];
  for (size_t k = 0; k < src.size(); k++) src[k] = 0.5 + (double)k;
  HostPart part[4];
  for (int k = 0; k < 4; k++) {
    out[k].assign(len[k], -1.0);
    part[k] = {mask >> k & 1 ? out[k].data() : nullptr, len[k]};
  }
  auto send = [](void *to, const void *from, size_t bytes, hipStream_t st) {
    return hipMemcpyAsync(to, from, bytes, hipMemcpyDeviceToHost, st);
  };
  if (staged_download(dev, s, src.data(), part, 4, send) != hipSuccess) return false;
  size_t at = 0;
  for (int k = 0; k < 4; k++)
    for (size_t q = 0; q < len[k]; q++, at++)
      if (out[k][q] != (mask >> k & 1 ? src[at] : -1.0)) return false;
  return true;
}

// handles on two devices, whichever is current at a download
static void devices() {
  stub::Stream s0, s1;
  s1.dev = 1;
  staging_open(0);
  staging_open(1);
  for (int cur = 0; cur < 2; cur++) {
    stub::device = cur;
    REQUIRE(download(0, &s0, 3000, 15));
    REQUIRE(download(1, &s1, 3000, 15));
    REQUIRE(stub::device == cur);
  }
  REQUIRE(stub::pinned == 4 && stub::events == 4);
  staging_close(0);
  REQUIRE(stub::pinned == 2 && stub::events == 2);
  REQUIRE(download(1, &s1, 100, 15));
  staging_close(1);
  REQUIRE(stub::pinned == 0 && stub::events == 0);
  // without buffers (no memory, a device past the table) the arrays come
  // straight
  staging_open(0);
  stub::out_of_memory = true;
  REQUIRE(download(0, &s0, 3000, 15));
  REQUIRE(download(kStageDevices, &s0, 3000, 15));
  staging_close(0);
}

// every choice of arrays, with totals before, at and behind a piece's edge:
// what is skipped is not moved
static void ranges() {
  stub::Stream s0;
  staging_open(0);
  const size_t piece = kStageBytes / sizeof(double);
  for (size_t n : {(size_t)1, piece / 53, piece / 15, piece / 15 + 1, 2 * piece / 18 + 1})
    for (int mask = 0; mask < 16; mask++) {
      stub::bytes = 0;
      REQUIRE(download(0, &s0, n, mask));
      size_t want = 0;
      const size_t len[4] = {3 * n, 15 * n, 15 * n, 20 * n};
      for (int k = 0; k < 4; k++) want += mask >> k & 1 ? len[k] * sizeof(double) : 0;
      REQUIRE(stub::bytes == want);
    }
  staging_close(0);
}

// a download that waits for its stream's work keeps no other one waiting
static void busy() {
  stub::Stream s0, s1;
  staging_open(0);
  s0.busy = true;
  bool ok0 = false, ok1 = false, done1 = false;
  std::thread a([&] { ok0 = download(0, &s0, 3000, 15); });
  std::this_thread::sleep_for(std::chrono::milliseconds(100));
  std::thread b([&] {
    ok1 = download(0, &s1, 3000, 15);
    std::lock_guard<std::mutex> lk(stub::mu);
    done1 = true;
    stub::cv.notify_all();
  });
  bool in_time;
  {
    std::unique_lock<std::mutex> lk(stub::mu);
    in_time = stub::cv.wait_for(lk, std::chrono::seconds(5), [&] { return done1; });
    s0.busy = false;
    stub::cv.notify_all();
  }
  a.join();
  b.join();
  staging_close(0);
  REQUIRE(in_time && ok0 && ok1);
}

int main(int argc, char **argv) {
  for (int k = 1; k < argc; k++) {
    const std::string name = argv[k];
    for (int e = 0; e < 2; e++) {
      stub::eager = e;
      stub::out_of_memory = false;
      if (name == "devices") devices();
      else if (name == "ranges") ranges();
      else if (name == "busy") busy();
      else return 2;
    }
    printf("%s ok\n", argv[k]);
  }
  return 0;
}
