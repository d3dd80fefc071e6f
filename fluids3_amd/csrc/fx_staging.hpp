// fx_staging.hpp -- host arrays to and from a stream through pinned memory.
//
// A copy to or from ordinary memory is one round trip of the runtime's own
// staging, 12 to 18 us however small, and waits for everything.  Here an
// upload is copied into pinned memory and queued: the caller's array is free
// again at once and nothing is waited for.  A download goes slot by slot, one
// being copied out while the next ones arrive; a long one is copied out by a
// few threads, because the link is faster than one thread that also faults in
// the pages of a new array.  Before / now, us: upload of 24 KB 15 / 3, of
// 1.2 MB 67 / 24 (55 to 65 with the wait); download of 24 KB 11 / 11, of 1.2 MB
// 78 / 72, of 4 MB 222 / 173, of 47 MB into new memory 4663 / 1862.  Longer
// uploads keep the runtime's copy, which reads the caller's pages in place
// (4 MB: 131 us, 162 so).
//
// One per system, on its stream, used by one thread at a time like the
// system itself; 12 MB of pinned memory, given back with it.  Where that is
// not to be had, arrays go through the runtime's copy after a wait.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <new>
#include <thread>

#include "fx_common.hpp"

namespace fx {

class Staging {
 public:
  Staging() = default;
  Staging(const Staging&) = delete;
  Staging& operator=(const Staging&) = delete;
  ~Staging() {
    for (hipEvent_t& e : m_ev)
      if (e) (void)hipEventDestroy(e);
    if (m_up) (void)hipHostFree(m_up);
    if (m_down) (void)hipHostFree(m_down);
  }

  void create(hipStream_t stream) {
    m_stream = stream;
    bool down = pin(&m_down, kSlots * kSlot);
    for (hipEvent_t& e : m_ev) down = down && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    m_slots = down;
    (void)pin(&m_up, kRing);
  }

  // Work queued on the stream after this sees dst filled.
  int up(void* dst, const void* src, size_t bytes, const char* who) {
    if (bytes > kUp || m_up == nullptr) {
      FX_TRY(drain(who));
      FX_HIP(hipMemcpyHtoD(dst, const_cast<void*>(src), bytes), who);
      return FX_OK;
    }
    if (m_used + bytes > kRing) FX_TRY(drain(who));
    for (size_t a = 0; a < bytes; a += kSlot) {
      const size_t n = std::min(kSlot, bytes - a);
      memcpy(m_up + m_used, static_cast<const char*>(src) + a, n);
      FX_HIP(hipMemcpyAsync(static_cast<char*>(dst) + a, m_up + m_used, n, hipMemcpyHostToDevice, m_stream), who);
      m_used += (n + 63) / 64 * 64;
    }
    return FX_OK;
  }

  // dst holds what src held after the work queued so far.
  int down(void* dst, const void* src, size_t bytes, const char* who) {
    char* from = static_cast<char*>(const_cast<void*>(src));
    char* to = static_cast<char*>(dst);
    if (bytes == 0) return drain(who);
    if (!m_slots) {
      FX_TRY(drain(who));
      FX_HIP(hipMemcpyDtoH(to, from, bytes), who);
      return FX_OK;
    }
    if (bytes > kDown) return down_long(to, from, bytes, who);
    const int chunks = (int)((bytes + kSlot - 1) / kSlot);
    auto size = [&](int k) { return std::min(kSlot, bytes - (size_t)k * kSlot); };
    for (int k = 0, queued = 0; k < chunks; k++) {
      for (; queued < chunks && queued < k + kSlots; queued++) {
        const int s = queued % kSlots;
        FX_HIP(hipMemcpyAsync(m_down + (size_t)s * kSlot, from + (size_t)queued * kSlot, size(queued),
                              hipMemcpyDeviceToHost, m_stream), who);
        if (chunks > 1) FX_HIP(hipEventRecord(m_ev[s], m_stream), who);
      }
      if (chunks > 1)
        FX_HIP(hipEventSynchronize(m_ev[k % kSlots]), who);
      else
        FX_HIP(hipStreamSynchronize(m_stream), who);
      memcpy(to + (size_t)k * kSlot, m_down + (size_t)(k % kSlots) * kSlot, size(k));
    }
    m_used = 0;  // every upload before them has been made
    return FX_OK;
  }

  // Everything queued on the stream is done.
  int drain(const char* who) {
    FX_HIP(hipStreamSynchronize(m_stream), who);
    m_used = 0;
    return FX_OK;
  }

 private:
  static constexpr int kSlots = 8;
  static constexpr size_t kSlot = 1 << 20;
  static constexpr size_t kRing = 4 << 20, kUp = 2 << 20, kDown = 4 << 20;

  static bool pin(char** p, size_t bytes) {
    if (hipHostMalloc(reinterpret_cast<void**>(p), bytes, hipHostMallocDefault) == hipSuccess) return true;
    (void)hipGetLastError();
    *p = nullptr;
    return false;
  }

  // As down, with the copies out of the slots made by kWorkers threads, which
  // take the chunks in turn: chunk c may be copied once ready > c, and its
  // slot is filled again once done[c] is set.
  int down_long(char* to, char* from, size_t bytes, const char* who) {
    constexpr int kWorkers = 3;
    FX_TRY(drain(who));  // no thread waits while the stream still computes
    const int chunks = (int)((bytes + kSlot - 1) / kSlot);
    auto size = [&](int k) { return std::min(kSlot, bytes - (size_t)k * kSlot); };
    std::unique_ptr<std::atomic<bool>[]> done(new (std::nothrow) std::atomic<bool>[chunks]());
    std::atomic<int> ready{0}, next{0};
    std::atomic<bool> stop{false};
    auto work = [&]() {
      for (int c = next.fetch_add(1); c < chunks; c = next.fetch_add(1)) {
        while (ready.load(std::memory_order_acquire) <= c) {
          if (stop.load(std::memory_order_relaxed)) return;
          std::this_thread::yield();
        }
        memcpy(to + (size_t)c * kSlot, m_down + (size_t)(c % kSlots) * kSlot, size(c));
        done[c].store(true, std::memory_order_release);
      }
    };
    std::thread worker[kWorkers];
    int workers = 0;
    try {
      if (done != nullptr)
        for (; workers < kWorkers; workers++) worker[workers] = std::thread(work);
    } catch (...) {  // no more threads or no memory for one: as many as could be started
    }
    if (workers == 0) {
      FX_HIP(hipMemcpyDtoH(to, from, bytes), who);
      return FX_OK;
    }
    hipError_t e = hipSuccess;
    for (int k = 0, queued = 0; k < chunks && e == hipSuccess; k++) {
      while (e == hipSuccess && queued < chunks && queued < k + kSlots) {
        const int s = queued % kSlots;
        if (queued >= kSlots && !done[queued - kSlots].load(std::memory_order_acquire)) {
          if (queued > k) break;  // wait for chunk k first
          std::this_thread::yield();
          continue;
        }
        e = hipMemcpyAsync(m_down + (size_t)s * kSlot, from + (size_t)queued * kSlot, size(queued),
                           hipMemcpyDeviceToHost, m_stream);
        if (e == hipSuccess) e = hipEventRecord(m_ev[s], m_stream);
        queued++;
      }
      if (e == hipSuccess) e = hipEventSynchronize(m_ev[k % kSlots]);
      if (e == hipSuccess) ready.store(k + 1, std::memory_order_release);
    }
    if (e != hipSuccess) stop.store(true);
    for (int w = 0; w < workers; w++) worker[w].join();
    if (e != hipSuccess) {
      (void)hipStreamSynchronize(m_stream);  // no copy into the slots is left under way
      return fx::hip_fail(e, who, "copy to the host");
    }
    return FX_OK;
  }

  hipStream_t m_stream = nullptr;
  char* m_up = nullptr;
  char* m_down = nullptr;
  size_t m_used = 0;  // of m_up, by copies that may not have been made
  bool m_slots = false;  // m_down and its events are there
  hipEvent_t m_ev[kSlots] = {};
};

}  // namespace fx
