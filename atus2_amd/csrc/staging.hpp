// staging.hpp -- device-to-host copies into ordinary (pageable) memory
// through pinned buffers of the library's own.
//
// The runtime's copy into fresh pageable memory takes 170 us for 1 MiB, 340 us
// for 2 MiB and 26 ms for 256 MiB (10 GB/s: one thread's memcpy, a third of it
// page faults).  Here the copy is cut into pieces that travel through pinned
// slots, so the transfer of one piece overlaps the memcpy of another, and
// large copies are memcpy'd by several threads, each with a slot of its own:
// 90 us, 120 us and 7.4 ms.  Up to 256 KiB the runtime's path is faster (26
// against 68 us), at 512 KiB the two are equal.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace atus_host {

class Staging {
 public:
  static constexpr int SLOTS = 4;
  static constexpr size_t SLOT = (size_t)4 << 20;   // largest piece
  static constexpr size_t PIECE = (size_t)256 << 10;  // smallest
  static constexpr size_t LEAST = (size_t)1 << 20;  // shorter copies take the runtime's path
  static constexpr size_t THREADED = (size_t)8 << 20;

  explicit Staging(int device) : device_(device) {}

  // the pool's memory lives while any context of its device does
  void ref() {
    std::lock_guard<std::mutex> l(m_);
    ++refs_;
  }
  void unref() {
    std::lock_guard<std::mutex> l(m_);
    if (--refs_ == 0) drop();
  }

  // copies `bytes` from device memory at src to dst after the work already on
  // `stream`; returns once dst holds them.  hipErrorNotReady: not done (a
  // short copy, another thread in the pool, no pinned memory): the caller
  // copies by itself.
  hipError_t to_host(void* dst, const void* src, size_t bytes, hipStream_t stream) {
    if (bytes < LEAST) return hipErrorNotReady;
    std::unique_lock<std::mutex> l(m_, std::try_to_lock);
    if (!l.owns_lock()) return hipErrorNotReady;
    // four pieces at least, so that transfer and memcpy overlap
    const size_t piece = std::min(SLOT, std::max(PIECE, (bytes / SLOTS + 4095) & ~(size_t)4095));
    const size_t n = (bytes + piece - 1) / piece;
    const int used = (int)std::min<size_t>(n, SLOTS);
    if (!reserve(used, piece)) return hipErrorNotReady;
    auto start = [&](size_t k, int s) {
      const size_t o = k * piece;
      hipError_t e = hipMemcpyAsync(slot_[s], (const char*)src + o, std::min(piece, bytes - o), hipMemcpyDeviceToHost,
                                    stream);
      return e == hipSuccess ? hipEventRecord(ev_[s], stream) : e;
    };
    auto finish = [&](size_t k, int s) {
      const size_t o = k * piece;
      const hipError_t e = hipEventSynchronize(ev_[s]);
      if (e == hipSuccess) memcpy((char*)dst + o, slot_[s], std::min(piece, bytes - o));
      return e;
    };
    hipError_t err = hipSuccess;
    if (bytes < THREADED) {
      for (size_t k = 0; k < (size_t)used && err == hipSuccess; ++k) err = start(k, (int)k);
      for (size_t k = 0; k < n && err == hipSuccess; ++k) {
        err = finish(k, (int)(k % SLOTS));
        if (err == hipSuccess && k + SLOTS < n) err = start(k + SLOTS, (int)(k % SLOTS));
      }
    } else {
      // piece k belongs to slot k % SLOTS and the thread that holds it
      std::atomic<int> first{(int)hipSuccess};
      auto work = [&](int s) {
        hipError_t e = hipSetDevice(device_);
        for (size_t k = s; k < n && e == hipSuccess; k += SLOTS) {
          e = start(k, s);
          if (e == hipSuccess) e = finish(k, s);
        }
        int ok = (int)hipSuccess;
        if (e != hipSuccess) first.compare_exchange_strong(ok, (int)e);
      };
      std::vector<std::thread> pool;
      int s = 1;
      try {
        for (; s < SLOTS; ++s) pool.emplace_back(work, s);
      } catch (...) {
        // no more threads: the caller's takes the rest
      }
      work(0);
      for (; s < SLOTS; ++s) work(s);
      for (std::thread& t : pool) t.join();
      err = (hipError_t)first.load();
    }
    // an error may leave transfers into the slots in flight
    if (err != hipSuccess) (void)hipStreamSynchronize(stream);
    return err;
  }

 private:
  bool reserve(int used, size_t piece) {
    for (int s = 0; s < used; ++s) {
      if (!ev_[s] && hipEventCreateWithFlags(&ev_[s], hipEventDisableTiming) != hipSuccess) {
        ev_[s] = nullptr;
        (void)hipGetLastError();
        return false;
      }
      if (cap_[s] >= piece) continue;
      if (slot_[s]) (void)hipHostFree(slot_[s]);
      slot_[s] = nullptr;
      cap_[s] = 0;
      size_t cap = PIECE;
      while (cap < piece) cap *= 2;
      if (hipHostMalloc(&slot_[s], cap, hipHostMallocDefault) != hipSuccess) {
        slot_[s] = nullptr;
        (void)hipGetLastError();
        return false;
      }
      cap_[s] = cap;
    }
    return true;
  }
  void drop() {
    for (int s = 0; s < SLOTS; ++s) {
      if (slot_[s]) (void)hipHostFree(slot_[s]);
      if (ev_[s]) (void)hipEventDestroy(ev_[s]);
      slot_[s] = nullptr;
      ev_[s] = nullptr;
      cap_[s] = 0;
    }
  }

  std::mutex m_;
  const int device_;
  int refs_ = 0;
  void* slot_[SLOTS] = {};
  size_t cap_[SLOTS] = {};
  hipEvent_t ev_[SLOTS] = {};
};

// the pool of a device (its slots and events, so that downloads from several
// devices neither wait for each other nor take turns in one pool's slots), or
// null; never destroyed: its memory goes with the device's last context, which
// may outlive static destruction
inline Staging* staging(int device) {
  constexpr int MOST = 64;
  static std::mutex m;
  static Staging* pool[MOST] = {};
  if (device < 0 || device >= MOST) return nullptr;
  std::lock_guard<std::mutex> l(m);
  if (!pool[device]) pool[device] = new (std::nothrow) Staging(device);
  return pool[device];
}

}  // namespace atus_host
