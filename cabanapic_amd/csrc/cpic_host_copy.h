// cpic_host_copy.h -- device memory into the caller's pageable host memory.
//
// The runtime's own pageable copy runs at 10.5 GB/s into memory that has just
// been allocated (one thread moves the data out of a staging buffer and takes
// the page faults): 7.9 ms for the 79 MB of fields of a 128^3 grid, an eighth
// of 24 steps.  Here 2 MB pieces of a pinned ring are filled while up to four
// threads empty it: 2.2 ms (36 GB/s; 50 MB 5.0 -> 1.5 ms), 1.7 into memory that is
// there (47 GB/s).  1 MB pieces reach 29 GB/s, one thread 14, six threads no more.
//
// A kernel fills them, not a copy engine: the GPU driver clears device memory that
// is given back with the copy engines, 30 ms for each GB, and what they copy
// meanwhile moves at 12 GB/s instead of 45 (79 MB 6.6 ms, by the kernel 1.7; a
// gradient of 64^3 x 32, 4 steps, by an Adjoint made for it 64 ms, by the kernel
// 38).
//
// The caller is one of the threads, and the only one below 16 MB, where others
// gain little (7 MB 0.45 against 0.5 ms) and cost much where the program's own
// threads, spinning after a parallel loop, use up the process's CPUs: gradients of
// 25x25x15 x 15 particles, whose owner rounds them with such a loop, took 1.8 or
// 4 ms a pass with four threads beside the caller, 1.8 always with the caller
// alone.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace cpic {

// n bytes of device memory into pinned memory, by a kernel on the stream.
hipError_t launch_to_pinned(void* pinned, const void* src, size_t n, hipStream_t stream);

// The pinned ring, one for the process: allocated by the first large download
// and given back with the last context.  A second thread's download at the
// same time takes the runtime's own path.
class HostRing {
 public:
  static constexpr size_t kPiece = 2u << 20;
  static constexpr int kPieces = 8;
  static constexpr int kThreads = 4;
  static constexpr size_t kSmall = 4u << 20;  // below this the plain copy is as fast
  static constexpr size_t kTiny = 16u << 10;  // to this the runtime's synchronous copy is
                                              // faster than one queued and waited for (12 us
                                              // and 21; beyond, both take the same time)

  static HostRing& get() {
    static HostRing ring;
    return ring;
  }
  // A context is opened (closed).  Neither waits for a download, which holds the
  // ring as long as the work queued before it runs: the last context to be closed
  // finds the ring free.
  void retain() {
    std::lock_guard<std::mutex> l(users_mutex_);
    ++users_;
  }
  void release() {
    std::lock_guard<std::mutex> l(users_mutex_);
    if (--users_ > 0) return;
    std::lock_guard<std::mutex> r(m_);
    if (ring_) (void)hipHostFree(ring_);
    ring_ = nullptr;
  }

  // n bytes of device memory into dst, after the work queued on the stream.  They
  // have arrived when the caller has waited for the stream: what the ring does not
  // take is left queued, so that the arrays of a download share one wait (the 8 of
  // 16 particles take 155 us, and 187 with a wait each).
  hipError_t copy(void* dst, const void* src, size_t n, hipStream_t stream) {
    std::unique_lock<std::mutex> l(m_, std::defer_lock);
    if (n < kSmall || pinned(dst) || !l.try_lock() || !ready())
      return hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, stream);
    return ringed((char*)dst, (const char*)src, n, stream);
  }

 private:
  std::mutex users_mutex_;  // taken before m_ where both are
  int users_ = 0;
  std::mutex m_;  // held while the ring is in use
  char* ring_ = nullptr;

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

  // Threads that empty the ring, the caller among them (each divides kPieces).
  static int threads_for(size_t n) { return n < (16u << 20) ? 1 : n < (32u << 20) ? 2 : kThreads; }

  // Piece i goes through slot i % kPieces and is thread i % threads's, which
  // empties the slot and then has it filled with the next piece of the slot, its
  // own too: the threads share nothing but the stream.
  hipError_t ringed(char* dst, const char* src, size_t n, hipStream_t stream) {
    const long pieces = (long)((n + kPiece - 1) / kPiece);
    const int threads = threads_for(n);
    hipEvent_t ev[kPieces] = {};
    int device = 0;
    hipError_t err = hipGetDevice(&device);
    for (int k = 0; k < kPieces && err == hipSuccess; ++k)
      err = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
    std::atomic<int> failure{(int)err};
    auto size = [&](long i) { return std::min(kPiece, n - (size_t)i * kPiece); };
    auto slot = [&](long i) { return ring_ + (size_t)(i % kPieces) * kPiece; };
    auto fill = [&](long i) {
      hipError_t e = launch_to_pinned(slot(i), src + (size_t)i * kPiece, size(i), stream);
      if (e == hipSuccess) e = hipEventRecord(ev[i % kPieces], stream);
      if (e != hipSuccess) failure = (int)e;
    };
    auto empty = [&](int t) {
      for (long i = t; i < pieces && failure == (int)hipSuccess; i += threads) {
        const hipError_t e = hipEventSynchronize(ev[i % kPieces]);
        if (e != hipSuccess) {
          failure = (int)e;
          return;
        }
        memcpy(dst + (size_t)i * kPiece, slot(i), size(i));
        if (i + kPieces < pieces) fill(i + kPieces);
      }
    };
    for (long i = 0; i < std::min<long>(pieces, kPieces) && failure == (int)hipSuccess; ++i) fill(i);
    std::vector<std::thread> pool;
    int started = 1;
    try {
      pool.reserve(threads);
      for (; started < threads; ++started)
        pool.emplace_back([&, t = started] {
          (void)hipSetDevice(device);
          empty(t);
        });
    } catch (...) {
      // no more threads to be had: the caller takes their pieces
    }
    empty(0);
    for (int t = started; t < threads; ++t) empty(t);
    for (auto& th : pool) th.join();
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    // (after a failure copies into the ring may still be in flight)
    if (failure != (int)hipSuccess) (void)hipStreamSynchronize(stream);
    return (hipError_t)failure.load();
  }
};

}  // namespace cpic
