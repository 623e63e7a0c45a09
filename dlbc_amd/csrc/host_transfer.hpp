// host_transfer.hpp -- fields and populations between device memory and the
// caller's pageable arrays.
//
// A transfer of more than one slot is cut into slots of 2 MB and dealt to a few
// threads, each with a pinned slot of its own: the copy engine moves one slot
// (57 GB/s) while the other threads copy theirs to or from the caller's array,
// page faults of a fresh array included.  134 MB into a fresh array: 12.8 ms as
// one copy into pageable memory, and 56 ms through an intermediate array, which
// was the way before; 4.2 ms here.  A transfer of one slot uses the calling
// thread alone.
//
// The slots belong to the process, at most kTransferKept of them while no
// transfer uses them, and are freed with the last context.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace dlbc {

constexpr size_t kSlotBytes = 2u << 20;
constexpr int kTransferThreads = 8, kTransferKept = 16;

// `device` is the calling thread's current one while this lives (ok: it is).
struct OnDevice {
  int before = -1;
  bool ok = true;
  explicit OnDevice(int device) {
    if (hipGetDevice(&before) != hipSuccess) before = -1;
    if (before == device)
      before = -1;  // nothing to give back
    else
      ok = hipSetDevice(device) == hipSuccess;
    if (!ok) (void)hipGetLastError();
  }
  ~OnDevice() {
    if (before >= 0) (void)hipSetDevice(before);
  }
  OnDevice(const OnDevice &) = delete;
  OnDevice &operator=(const OnDevice &) = delete;
};

struct PinnedSlot {
  void *p = nullptr;
  hipEvent_t done = nullptr;
  int device = 0;
};

// Slots that no transfer uses, and the contexts that may.
struct SlotPool {
  std::mutex mu;
  std::vector<PinnedSlot> idle;
  int users = 0;

  SlotPool() { idle.reserve(kTransferKept); }  // (give() is called from threads and never throws)
  static void drop(PinnedSlot s) {
    if (s.done) (void)hipEventDestroy(s.done);
    if (s.p) (void)hipHostFree(s.p);
  }
  void enter() {
    std::lock_guard<std::mutex> lock(mu);
    ++users;
  }
  void leave() {
    std::lock_guard<std::mutex> lock(mu);
    if (--users > 0) return;
    for (auto &s : idle) drop(s);
    idle.clear();
  }
  // A slot for `device`; p is null where there is no memory.
  PinnedSlot take(int device) {
    {
      std::lock_guard<std::mutex> lock(mu);
      for (size_t k = idle.size(); k-- > 0;)
        if (idle[k].device == device) {
          const PinnedSlot s = idle[k];
          idle.erase(idle.begin() + (std::ptrdiff_t)k);
          return s;
        }
    }
    PinnedSlot s;
    s.device = device;
    const OnDevice on(device);
    if (!on.ok || hipHostMalloc(&s.p, kSlotBytes, hipHostMallocPortable) != hipSuccess ||
        hipEventCreateWithFlags(&s.done, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      drop(s);
      return PinnedSlot{};
    }
    return s;
  }
  void give(PinnedSlot s) {
    if (!s.p) return;
    {
      std::lock_guard<std::mutex> lock(mu);
      if (users > 0 && idle.size() < (size_t)kTransferKept) {
        idle.push_back(s);
        return;
      }
    }
    drop(s);
  }
};

inline SlotPool &slot_pool() {
  static SlotPool *pool = new SlotPool();  // (never destroyed: the runtime may be gone by then)
  return *pool;
}

// work(slot, k) for the parts k = 0 .. parts-1 of a transfer on `stream`, each
// thread with a slot of its own.  Returns the first error; without a pinned slot
// hipErrorOutOfMemory before any part is done.
template <class Work>
inline hipError_t transfer_parts(int device, hipStream_t stream, int parts, Work work) {
  PinnedSlot mine = slot_pool().take(device);
  if (!mine.p) return hipErrorOutOfMemory;
  std::atomic<int> next{0};
  std::atomic<int> err{(int)hipSuccess};
  auto run = [&](PinnedSlot &s) {
    for (int k; err.load() == hipSuccess && (k = next.fetch_add(1)) < parts;) {
      const hipError_t e = work(s, k);
      if (e == hipSuccess) continue;
      err.store((int)e);
      // a copy may be under way in the slot: where that cannot be waited for, the
      // slot is left alone for good
      if (hipStreamSynchronize(stream) != hipSuccess) s = PinnedSlot{};
      return;
    }
  };
  std::vector<std::thread> threads;
  try {
    for (int t = 1; t < std::min(parts, kTransferThreads); ++t)
      threads.emplace_back([&, device] {
        if (hipSetDevice(device) != hipSuccess) return;
        PinnedSlot s = slot_pool().take(device);
        if (!s.p) return;  // the other threads do its parts
        run(s);
        slot_pool().give(s);
      });
  } catch (const std::exception &) {  // no thread, no memory: the ones there are will do
  }
  run(mine);
  for (auto &t : threads) t.join();
  slot_pool().give(mine);
  return (hipError_t)err.load();
}

// Device memory to the host: put(offset, data, bytes) takes the bytes at
// `offset` of dev; called from several threads for disjoint ranges.
template <class Put>
inline hipError_t transfer_down(int device, hipStream_t stream, const void *dev, size_t bytes,
                                Put put) {
  const int parts = (int)((bytes + kSlotBytes - 1) / kSlotBytes);
  return transfer_parts(device, stream, parts, [&](const PinnedSlot &s, int k) {
    const size_t o = (size_t)k * kSlotBytes, n = std::min(kSlotBytes, bytes - o);
    hipError_t e = hipMemcpyAsync(s.p, static_cast<const char *>(dev) + o, n,
                                  hipMemcpyDeviceToHost, stream);
    if (e == hipSuccess) e = hipEventRecord(s.done, stream);
    if (e == hipSuccess) e = hipEventSynchronize(s.done);
    if (e == hipSuccess) put(o, static_cast<const char *>(s.p), n);
    return e;
  });
}

// The host to device memory: get(offset, data, bytes) fills the bytes at
// `offset`.  Every copy has ended when it returns.
template <class Get>
inline hipError_t transfer_up(int device, hipStream_t stream, void *dev, size_t bytes, Get get) {
  const int parts = (int)((bytes + kSlotBytes - 1) / kSlotBytes);
  return transfer_parts(device, stream, parts, [&](const PinnedSlot &s, int k) {
    const size_t o = (size_t)k * kSlotBytes, n = std::min(kSlotBytes, bytes - o);
    get(o, static_cast<char *>(s.p), n);
    hipError_t e = hipMemcpyAsync(static_cast<char *>(dev) + o, s.p, n, hipMemcpyHostToDevice,
                                  stream);
    if (e == hipSuccess) e = hipEventRecord(s.done, stream);
    if (e == hipSuccess) e = hipEventSynchronize(s.done);
    return e;
  });
}

}  // namespace dlbc
