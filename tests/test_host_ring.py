"""The pinned download ring against a stand-in for the runtime, on the CPU: a
download that waits for the work queued before it keeps no other thread from
opening or closing a context, one too small for the ring is left queued, the data
arrive whole, and the ring is given back with the last context."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cabanapic_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <condition_variable>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <mutex>
enum hipError_t { hipSuccess, hipErrorInvalidValue };
enum { hipMemcpyDeviceToHost, hipEventDisableTiming, hipHostMallocPortable };
enum hipMemoryType { hipMemoryTypeUnregistered, hipMemoryTypeHost };
struct hipPointerAttribute_t { hipMemoryType type; };
typedef void* hipStream_t;
typedef void* hipEvent_t;
// the one stream: its work is done when `open` says so
struct Gate {
  std::mutex m;
  std::condition_variable cv;
  bool open = false;
  int waiting = 0, allocated = 0;
  void pass() {
    std::unique_lock<std::mutex> l(m);
    ++waiting;
    cv.notify_all();
    cv.wait(l, [&] { return open; });
  }
};
inline Gate gate;
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
  memcpy(d, s, n);
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return gate.pass(), hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return gate.pass(), hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) { return *e = &gate, hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) {
  return hipErrorInvalidValue;
}
inline hipError_t hipHostMalloc(void** p, size_t n, int) {
  ++gate.allocated;
  *p = malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  --gate.allocated;
  free(p);
  return hipSuccess;
}
"""

PROGRAM = r"""
#include "cpic_host_copy.h"
#include <chrono>
#include <cstdio>
#include <future>
hipError_t cpic::launch_to_pinned(void* d, const void* s, size_t n, hipStream_t st) {
  return hipMemcpyAsync(d, s, n, hipMemcpyDeviceToHost, st);
}
int main(int, char** argv) {
  const size_t n = atol(argv[1]);
  std::vector<char> src(n), dst(n), small(4096);
  for (size_t i = 0; i < n; ++i) src[i] = (char)(i * 31 + i / 4096);
  cpic::HostRing& ring = cpic::HostRing::get();
  ring.retain();
  auto queued = std::async(std::launch::async,
                           [&] { return ring.copy(small.data(), src.data(), small.size(), nullptr); });
  const bool at_once = queued.wait_for(std::chrono::seconds(10)) == std::future_status::ready;
  auto download = std::async(std::launch::async, [&] { return ring.copy(dst.data(), src.data(), n, nullptr); });
  {
    std::unique_lock<std::mutex> l(gate.m);
    gate.cv.wait(l, [&] { return gate.waiting > 0; });
  }
  auto other = std::async(std::launch::async, [&] { ring.retain(); ring.release(); });
  const bool free = other.wait_for(std::chrono::seconds(10)) == std::future_status::ready;
  {
    std::lock_guard<std::mutex> l(gate.m);
    gate.open = true;
    gate.cv.notify_all();
  }
  const bool ok = download.get() == hipSuccess && queued.get() == hipSuccess &&
                  memcmp(small.data(), src.data(), small.size()) == 0;
  other.get();
  const int held = gate.allocated;
  ring.release();
  printf("%d %d %d %d %d %d\n", at_once, free, ok, src == dst, held, gate.allocated);
}
"""


# one thread, two and four; a whole number of pieces, and not
@pytest.mark.parametrize("size", [(4 << 20) + 5, 18 << 20, (40 << 20) - 3])
def test_contexts_come_and_go_during_a_download(tmp_path, size):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "main.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "ring")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-pthread", "-I", str(tmp_path), "-I", CSRC,
                    "-o", exe, str(tmp_path / "main.cpp")], check=True)
    out = subprocess.run([exe, str(size)], check=True, capture_output=True, text=True, timeout=60)
    # nothing waited, success, the right bytes, one ring held and then none
    assert out.stdout.split() == ["1", "1", "1", "1", "1", "0"]
