// Host side of whole snapshots: a ring of pinned host slots and the loop that runs a snapshot's
// pieces through them. A kernel writes a slot (or reads it) over the bus, copying threads move it to
// (from) the caller's memory, so both run at once and the page faults of fresh memory are shared
// out. One ring per process, given back when the last cache goes; one transfer has it at a time,
// and a transfer that finds it taken does not wait for it (the other's stream may be long busy).
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

namespace bg {

struct SnapshotRing {
  static constexpr int kSlots = 8;
  static constexpr size_t kSlotBytes = (size_t)2 << 20;
  std::mutex mu;
  char* host = nullptr;
  char* dev = nullptr;
  hipEvent_t ev[kSlots] = {};
  int device = -1;  // of the events

  // The ring for one transfer on the current device, held as long as the lock; an empty lock when
  // another transfer has it or its slots cannot be had.
  std::unique_lock<std::mutex> take() {
    std::unique_lock<std::mutex> lock(mu, std::try_to_lock);
    if (lock && ensure() != hipSuccess) {
      (void)hipGetLastError();
      lock.unlock();
    }
    return lock;
  }

  void drop() {
    std::lock_guard<std::mutex> lock(mu);
    give_back();
  }

 private:
  void drop_events() {
    for (hipEvent_t& e : ev)
      if (e) {
        (void)hipEventDestroy(e);
        e = nullptr;
      }
    device = -1;
  }
  void give_back() {
    drop_events();
    if (host) (void)hipHostFree(host);
    host = dev = nullptr;
  }
  // The slots serve every device. Events are the device's that was current at their creation and
  // can be recorded on its streams alone, so it is that device, not a cache's, they are kept for.
  hipError_t ensure() {
    int d = 0;
    hipError_t e = hipGetDevice(&d);
    if (e != hipSuccess || (host && device == d)) return e;
    drop_events();
    if (!host) {
      e = hipHostMalloc((void**)&host, kSlots * kSlotBytes, hipHostMallocMapped | hipHostMallocPortable | hipHostMallocCoherent);
      if (e != hipSuccess) host = nullptr;
    }
    if (e == hipSuccess) e = hipHostGetDevicePointer((void**)&dev, host, 0);
    for (hipEvent_t& x : ev)
      if (e == hipSuccess) e = hipEventCreateWithFlags(&x, hipEventDisableTiming);
    if (e != hipSuccess) give_back();
    else device = d;
    return e;
  }
};

// Runs n pieces through the slots. issue(i): main thread, enqueues piece i's kernel and records its
// event; copy(i): any thread, moves piece i between its slot and the caller. Export copies a piece
// once its event has passed; import copies it first, once the event of the slot's last piece has.
template <typename Issue, typename Copy>
hipError_t snapshot_run(SnapshotRing& ring, int n, bool import_, Issue issue, Copy copy) {
  constexpr int kSlots = SnapshotRing::kSlots;
  std::mutex mu;
  std::condition_variable cv;
  int issued = 0;                    // pieces whose event is recorded
  std::vector<char> copied(n, 0);
  hipError_t err = hipSuccess;
  auto wait_event = [&](int i) {
    const hipError_t e = hipEventSynchronize(ring.ev[i % kSlots]);
    if (e != hipSuccess) {
      std::lock_guard<std::mutex> l(mu);
      err = e;
    }
  };
  auto one = [&](int i) {  // piece i's copy, on a copying thread
    const int after = import_ ? i - kSlots : i;  // whose event must have passed
    if (after >= 0) {
      {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [&] { return issued > after || err != hipSuccess; });
        if (err != hipSuccess) return;
      }
      wait_event(after);
    }
    copy(i);
    std::lock_guard<std::mutex> l(mu);
    copied[i] = 1;
    cv.notify_all();
  };
  std::vector<std::thread> threads;
  const int want = std::min(4, n);
  int workers = 0;
  std::atomic<int> next{0};
  auto work = [&] {
    for (int i = next.fetch_add(1); i < n; i = next.fetch_add(1)) one(i);
  };
  try {
    threads.reserve(want);
    for (; workers < want; workers++) threads.emplace_back(work);
  } catch (...) {
    // as many as there are; none: the copies run here
  }
  for (int i = 0; i < n; i++) {
    const int need = import_ ? i : i - kSlots;  // the copy that must be done before the kernel
    if (need >= 0 && threads.empty() && import_) one(i);
    if (need >= 0) {
      std::unique_lock<std::mutex> l(mu);
      cv.wait(l, [&] { return copied[need] || err != hipSuccess; });
      if (err != hipSuccess) break;
    }
    const hipError_t e = issue(i);
    {
      std::lock_guard<std::mutex> l(mu);
      if (e != hipSuccess) err = e;
      else issued = i + 1;
      cv.notify_all();
    }
    if (e != hipSuccess) break;
    if (threads.empty() && !import_) one(i);
  }
  {
    std::lock_guard<std::mutex> l(mu);
    cv.notify_all();
  }
  for (std::thread& t : threads) t.join();
  return err;
}

}  // namespace bg
