// cpic_host_copy.h -- device memory into the caller's pageable host memory.
//
// The runtime's own pageable copy runs at 10.5 GB/s into memory that has just
// been allocated (one thread moves the data out of a staging buffer and takes
// the page faults): 7.9 ms for the 79 MB of fields of a 128^3 grid, an eighth
// of 24 steps.  Here the copy engine fills 2 MB pieces of a pinned ring while
// four threads empty it: 2.2 ms (36 GB/s; 10 MB 0.99 -> 0.46 ms, 50 MB 5.0 ->
// 1.5 ms).  1 MB pieces reach 29 GB/s, one thread 14, six threads no more.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace cpic {

// The pinned ring, one for the process: allocated by the first large download
// and given back with the last context.  A second thread's download at the
// same time takes the runtime's own path.
class HostRing {
 public:
  static constexpr size_t kPiece = 2u << 20;
  static constexpr int kPieces = 8;
  static constexpr int kThreads = 4;
  static constexpr size_t kSmall = 4u << 20;  // below this the plain copy is as fast

  static HostRing& get() {
    static HostRing ring;
    return ring;
  }
  void retain() {
    std::lock_guard<std::mutex> l(m_);
    ++users_;
  }
  void release() {
    std::lock_guard<std::mutex> l(m_);
    if (--users_ == 0 && ring_) {
      (void)hipHostFree(ring_);
      ring_ = nullptr;
    }
  }

  // n bytes of device memory into dst, after the work queued on the stream;
  // returns when they have arrived.
  hipError_t copy(void* dst, const void* src, size_t n, hipStream_t stream) {
    std::unique_lock<std::mutex> l(m_, std::defer_lock);
    if (n < kSmall || pinned(dst) || !l.try_lock() || !ready()) return plain(dst, src, n, stream);
    return ringed((char*)dst, (const char*)src, n, stream);
  }

 private:
  std::mutex m_;
  int users_ = 0;
  char* ring_ = nullptr;

  static hipError_t plain(void* dst, const void* src, size_t n, hipStream_t stream) {
    const hipError_t e = hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, stream);
    return e != hipSuccess ? e : hipStreamSynchronize(stream);
  }
  static bool pinned(const void* p) {
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
      (void)hipGetLastError();  // pageable memory is no error here
      return false;
    }
    return at.type != hipMemoryTypeUnregistered;
  }
  bool ready() {
    if (!ring_ &&
        hipHostMalloc((void**)&ring_, kPiece * kPieces, hipHostMallocPortable) != hipSuccess) {
      (void)hipGetLastError();
      ring_ = nullptr;
    }
    return ring_ != nullptr;
  }

  hipError_t ringed(char* dst, const char* src, size_t n, hipStream_t stream) {
    const long pieces = (long)((n + kPiece - 1) / kPiece);
    auto size = [&](long i) { return std::min(kPiece, n - (size_t)i * kPiece); };
    std::vector<std::thread> pool;
    pool.reserve(kThreads);
    hipEvent_t ev[kPieces] = {};
    int device = 0;
    hipError_t err = hipGetDevice(&device);
    for (int k = 0; k < kPieces && err == hipSuccess; ++k)
      err = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
    // piece i is in slot i % kPieces; queued: pieces handed to the copy engine,
    // emptied[t]: pieces that thread t (i % threads == t) has copied out.  A
    // piece is counted whatever became of it, so that nobody waits for ever.
    std::atomic<long> queued{0};
    std::atomic<long> emptied[kThreads];
    for (auto& e : emptied) e = 0;
    std::atomic<int> failure{(int)hipSuccess};
    auto empty = [&](int t) {
      (void)hipSetDevice(device);
      for (long i = t; i < pieces; i += kThreads) {
        while (queued.load(std::memory_order_acquire) <= i) std::this_thread::yield();
        if (failure.load() == (int)hipSuccess) {
          const hipError_t e = hipEventSynchronize(ev[i % kPieces]);
          if (e == hipSuccess)
            memcpy(dst + (size_t)i * kPiece, ring_ + (size_t)(i % kPieces) * kPiece, size(i));
          else
            failure = (int)e;
        }
        emptied[t].fetch_add(1, std::memory_order_release);
      }
    };
    if (err == hipSuccess) {
      try {
        for (int t = 0; t < kThreads; ++t) pool.emplace_back(empty, t);
      } catch (...) {
        // no threads to be had: those that started are let run dry
        failure = (int)hipErrorOutOfMemory;
        queued = pieces;
        for (auto& th : pool) th.join();
        for (hipEvent_t e : ev) (void)hipEventDestroy(e);
        return plain(dst, src, n, stream);
      }
      for (long i = 0; i < pieces; ++i) {
        const long before = i - kPieces;  // the piece that had the slot
        if (before >= 0)
          while (emptied[before % kThreads].load(std::memory_order_acquire) <= before / kThreads)
            std::this_thread::yield();
        if (failure.load() == (int)hipSuccess) {
          hipError_t e = hipMemcpyAsync(ring_ + (size_t)(i % kPieces) * kPiece,
                                        src + (size_t)i * kPiece, size(i), hipMemcpyDeviceToHost,
                                        stream);
          if (e == hipSuccess) e = hipEventRecord(ev[i % kPieces], stream);
          if (e != hipSuccess) failure = (int)e;
        }
        queued.store(i + 1, std::memory_order_release);
      }
      for (auto& th : pool) th.join();
      err = (hipError_t)failure.load();
    }
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    // (after a failure copies into the ring may still be in flight)
    if (err != hipSuccess) (void)hipStreamSynchronize(stream);
    return err;
  }
};

}  // namespace cpic
