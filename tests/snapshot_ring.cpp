// Host test of csrc/bg_snapshot.h over a stand-in for the HIP calls it makes: events that remember
// their device, allocations that can be made to fail. Prints "ok".
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "bg_snapshot.h"

static int g_device = 0, g_allocs = 0, g_live = 0;
static bool g_no_memory = false;
struct Event {
  int device;
};

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (g_no_memory) return hipErrorOutOfMemory;
  g_allocs++, g_live++;
  *p = malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  g_live--;
  free(p);
  return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
  *d = h;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  g_live++;
  *e = (hipEvent_t) new Event{g_device};
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  g_live--;
  delete (Event*)e;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDevice(int* d) {
  *d = g_device;
  return hipSuccess;
}
}

#define CHECK(x)                                         \
  do {                                                   \
    if (!(x)) {                                          \
      printf("line %d: %s\n", __LINE__, #x);             \
      return 1;                                          \
    }                                                    \
  } while (0)

static bg::SnapshotRing ring;

// a snapshot of n pieces of one slot each, out of and into `data`, kernels being plain copies
static bool round_trip(int n) {
  std::vector<char> from(n), to(n), back(n);
  for (int i = 0; i < n; i++) from[i] = (char)(i * 7 + 1);
  char* s = ring.host;
  const size_t B = bg::SnapshotRing::kSlotBytes;
  const int K = bg::SnapshotRing::kSlots;
  hipError_t e = bg::snapshot_run(ring, n, false, [&](int i) { return s[i % K * B] = from[i], hipSuccess; },
                                  [&](int i) { to[i] = s[i % K * B]; });
  if (e != hipSuccess || to != from) return false;
  e = bg::snapshot_run(ring, n, true, [&](int i) { return back[i] = s[i % K * B], hipSuccess; },
                       [&](int i) { s[i % K * B] = to[i]; });
  return e == hipSuccess && back == from;
}

int main() {
  {
    auto lock = ring.take();
    CHECK(lock);
    for (int n : {1, 7, 8, 9, 61}) CHECK(round_trip(n));
    // a kernel that cannot be launched ends the transfer with its error
    CHECK(bg::snapshot_run(ring, 30, false, [](int i) { return i < 11 ? hipSuccess : hipErrorInvalidValue; }, [](int) {}) ==
          hipErrorInvalidValue);
    // the ring is taken: another transfer is told so at once
    bool other = true;
    const auto t0 = std::chrono::steady_clock::now();
    std::thread([&] { other = (bool)ring.take(); }).join();
    CHECK(!other && std::chrono::steady_clock::now() - t0 < std::chrono::seconds(5));
  }
  CHECK(ring.take() && g_allocs == 1);
  // another device current: its own events, the same slots, and back
  for (int d : {1, 1, 0}) {
    g_device = d;
    CHECK(ring.take());
    for (hipEvent_t e : ring.ev) CHECK(((Event*)e)->device == d);
  }
  CHECK(g_allocs == 1);
  ring.drop();
  CHECK(g_live == 0);
  g_no_memory = true;
  CHECK(!ring.take() && g_live == 0);
  g_no_memory = false;
  CHECK(ring.take());
  ring.drop();
  CHECK(g_live == 0);
  printf("ok\n");
  return 0;
}
