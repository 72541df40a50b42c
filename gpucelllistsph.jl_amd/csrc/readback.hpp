// Copies from the device into a caller's (pageable) memory.
//
// A copy straight into pageable memory runs at ~4 GB/s here, most of it the
// first touch of fresh pages.  Here the device writes chunks into a small set of
// page-locked slots (57 GB/s) while up to four host threads move finished
// chunks on, page faults included.
#pragma once

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "gclsph_internal.hpp"

namespace gclsph {

// The stream's device is the thread's current one within the scope: an event can
// be recorded on a stream of its own device only, and a thread that reads results
// may have another one current (a new thread has device 0).
class OnDeviceOf {
 public:
  explicit OnDeviceOf(hipStream_t st) {
    GCL_HIP(hipStreamGetDevice(st, &device));
    GCL_HIP(hipGetDevice(&before_));
    if (before_ != device) GCL_HIP(hipSetDevice(device));
  }
  ~OnDeviceOf() {
    if (before_ != device) (void)hipSetDevice(before_);
  }
  OnDeviceOf(const OnDeviceOf&) = delete;
  OnDeviceOf& operator=(const OnDeviceOf&) = delete;
  int device = 0;

 private:
  int before_ = 0;
};

// The page-locked slots: a set of them for each copy that runs.  Up to kKept sets
// stay for the next copies, of any object and device; the last object (Ref) to
// go frees them.  The lock is held to take a set and to give it back only.
class HostSlots {
 public:
  static constexpr size_t kSlot = size_t(1) << 20;
  static constexpr int kThreads = 4, kSlots = 2 * kThreads, kKept = 4;

  // Held by every object that may copy.
  struct Ref {
    Ref() {
      std::lock_guard<std::mutex> l(self().mutex_);
      ++self().refs_;
    }
    ~Ref() {
      HostSlots& s = self();
      std::lock_guard<std::mutex> l(s.mutex_);
      if (--s.refs_ > 0) return;
      while (s.kept_ > 0) (void)hipHostFree(s.free_[--s.kept_]);
    }
    Ref(const Ref&) = delete;
    Ref& operator=(const Ref&) = delete;
  };

  // out[0..bytes) from the device: fill(slot, offset, len) enqueues on st the
  // writing of bytes [offset, offset + len) to the page-locked slot (it may be
  // called from several threads, one chunk each).  Returns when out is complete.
  template <typename Fill>
  static void copy_out(void* out, size_t bytes, hipStream_t st, const Fill& fill) {
    if (bytes == 0) return;
    const OnDeviceOf on(st);
    const Set set;
    char* dst = static_cast<char*>(out);
    if (bytes <= kSlot) {
      fill(set.mem, size_t(0), bytes);
      GCL_HIP(hipStreamSynchronize(st));
      std::memcpy(dst, set.mem, bytes);
      return;
    }
    const size_t chunks = (bytes + kSlot - 1) / kSlot;
    // a thread pays from about a megabyte on (~20 us to start one)
    const int threads = int(std::min<size_t>(kThreads, (chunks + 1) / 2));
    std::exception_ptr failed;  // the first failure of a thread
    std::mutex failed_mutex;
    auto work = [&](int t) noexcept {
      hipEvent_t ev[2] = {nullptr, nullptr};
      try {
        GCL_HIP(hipSetDevice(on.device));
        for (auto& e : ev) GCL_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        auto start = [&](size_t c, int k) {
          fill(set.mem + kSlot * size_t(2 * t + k), c * kSlot, std::min(kSlot, bytes - c * kSlot));
          GCL_HIP(hipEventRecord(ev[k], st));
        };
        for (int k = 0; k < 2; ++k)
          if (size_t(t + k * threads) < chunks) start(size_t(t + k * threads), k);
        int k = 0;
        for (size_t c = size_t(t); c < chunks; c += size_t(threads), k ^= 1) {
          GCL_HIP(hipEventSynchronize(ev[k]));
          std::memcpy(dst + c * kSlot, set.mem + kSlot * size_t(2 * t + k), std::min(kSlot, bytes - c * kSlot));
          if (c + 2 * size_t(threads) < chunks) start(c + 2 * size_t(threads), k);
        }
      } catch (...) {
        std::lock_guard<std::mutex> l(failed_mutex);
        if (!failed) failed = std::current_exception();
      }
      for (auto& e : ev)
        if (e) (void)hipEventDestroy(e);
    };
    std::vector<std::thread> pool;
    int started = 1;
    try {
      for (; started < threads; ++started) pool.emplace_back(work, started);
    } catch (...) {  // no more threads to be had: their share is done here
    }
    work(0);
    for (auto& t : pool) t.join();
    for (int t = started; t < threads; ++t) work(t);
    const hipError_t end = hipStreamSynchronize(st);  // the slots are free again, also after a failure
    if (failed) std::rethrow_exception(failed);
    GCL_HIP(end);
  }

 private:
  // A copy's own slots.
  struct Set {
    char* mem = nullptr;
    Set() {
      HostSlots& s = self();
      {
        std::lock_guard<std::mutex> l(s.mutex_);
        if (s.kept_ > 0) mem = s.free_[--s.kept_];
      }
      if (mem) return;
      void* p = nullptr;
      GCL_HIP(hipHostMalloc(&p, kSlot * kSlots, hipHostMallocPortable));
      mem = static_cast<char*>(p);
    }
    ~Set() {
      HostSlots& s = self();
      {
        std::lock_guard<std::mutex> l(s.mutex_);
        if (s.refs_ > 0 && s.kept_ < kKept) {
          s.free_[s.kept_++] = mem;
          return;
        }
      }
      (void)hipHostFree(mem);
    }
    Set(const Set&) = delete;
    Set& operator=(const Set&) = delete;
  };

  static HostSlots& self() {
    static HostSlots s;
    return s;
  }
  std::mutex mutex_;
  int refs_ = 0, kept_ = 0;
  char* free_[kKept] = {};
};

}  // namespace gclsph
