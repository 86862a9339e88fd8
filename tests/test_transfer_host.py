"""The threaded copies between host arrays and the device (fvwb_transfer.h) on
the CPU: the header is compiled against a small model of the runtime in which a
copy moves its bytes only when the stream gets to it, so that a slot written
before its transfer is done gives wrong data."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fvm-source-wb_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <mutex>
enum hipError_t { hipSuccess, hipErrorInvalidValue, hipErrorOutOfMemory, hipErrorInvalidHandle };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum hipMemoryType { hipMemoryTypeUnregistered, hipMemoryTypeHost };
enum { hipEventDisableTiming = 2, hipHostMallocDefault = 0 };
struct hipPointerAttribute_t { hipMemoryType type; };
struct Event { int dev; long mark; };
struct Op { void* dst; const void* src; size_t n; };
struct Stream { int dev; std::deque<Op> ops; long done, queued; };
typedef Event* hipEvent_t;
typedef Stream* hipStream_t;
inline std::recursive_mutex mu;
inline Stream* the_stream = nullptr;
inline thread_local int current = 0;
inline size_t pinned = 0, pinned_most = 0, runtime_copies = 0;
inline const void* known_array = nullptr;
inline bool pin_fails = false;
#define LOCK std::lock_guard<std::recursive_mutex> lock(mu)
inline void run(Stream* s, long to) {
  for (; s->done < to; ++s->done) {
    std::memcpy(s->ops.front().dst, s->ops.front().src, s->ops.front().n);
    s->ops.pop_front();
  }
}
inline hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, int* d) { *d = s->dev; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  a->type = hipMemoryTypeHost;
  return p == known_array ? hipSuccess : hipErrorInvalidValue;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { LOCK; *e = new Event{current, 0}; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  LOCK;
  if (pin_fails) return hipErrorOutOfMemory;
  size_t* b = (size_t*)std::malloc(n + 64);
  *b = n;
  *p = b + 8;
  pinned += n;
  if (pinned > pinned_most) pinned_most = pinned;
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  LOCK;
  size_t* b = (size_t*)p - 8;
  pinned -= *b;
  std::memset(p, 0x5a, *b);                 // a transfer still under way would show
  std::free(b);
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  LOCK;
  if (n > (4u << 20)) ++runtime_copies;
  st->ops.push_back({d, s, n});
  ++st->queued;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  LOCK;
  if (e->dev != s->dev) return hipErrorInvalidHandle;
  e->mark = s->queued;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) { LOCK; run(the_stream, e->mark); return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s) { LOCK; run(s, s->queued); return hipSuccess; }
"""

MAIN = r"""
#include <cstdio>
#include <new>
#include <string>
#include <vector>
#include "fvwb_transfer.h"
static thread_local int new_countdown = -1;         // this thread's allocation that fails
void* operator new(size_t n) {
  if (new_countdown >= 0 && new_countdown-- == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

int main(int argc, char** argv) {
  const std::string what = argv[1];
  Stream st{what == "device" ? 1 : 0, {}, 0, 0};
  the_stream = &st;
  const size_t MB = 1 << 20;
  pin_fails = what == "unpinned";
  unsigned seed = 1;
  size_t most = 0;
  {
    fvwb_xfer::Staging s;
    for (size_t bytes : {size_t(3 * MB), size_t(9 * MB + 8), size_t(34 * MB - 24), size_t(150 * MB + 40), size_t(40 * MB)}) {
      std::vector<unsigned> up(bytes / 4), mid(bytes / 4), down(bytes / 4);
      for (auto& x : up) x = seed = seed * 1664525u + 1013904223u;
      for (int k = 0; k < 3; ++k) {                 // the k-th allocation of a copy fails
        std::fill(mid.begin(), mid.end(), 0u);
        std::fill(down.begin(), down.end(), 0u);
        const bool fail = what == "memory" && s.slots;
        if (fail) new_countdown = k;
        hipError_t e = fvwb_xfer::to_device(s, mid.data(), up.data(), bytes, &st);
        new_countdown = -1;
        if (e != hipSuccess) return std::printf("up %zu: error %d\n", bytes, e), 1;
        if (fail) new_countdown = k;
        e = fvwb_xfer::to_host(s, down.data(), mid.data(), bytes, &st);
        new_countdown = -1;
        if (e != hipSuccess) return std::printf("down %zu: error %d\n", bytes, e), 1;
        hipStreamSynchronize(&st);
        // what is pinned: about half the largest copy, at most 32 MB
        most = std::max(most, bytes < 8 * MB ? 0 : std::min(bytes / 2 + MB, 32 * MB));
        if (pinned > most) return std::printf("%zu bytes: %zu pinned\n", bytes, pinned), 1;
        if (up != down) return std::printf("%zu bytes differ\n", bytes), 1;
        if (current != 0) return std::printf("the caller's device changed\n"), 1;
      }
    }
    if (what == "known") {
      std::vector<char> a(64 * MB, 1), b(64 * MB);
      known_array = a.data();
      const size_t before = runtime_copies;
      if (fvwb_xfer::to_device(s, b.data(), a.data(), 64 * MB, &st) != hipSuccess || runtime_copies != before + 1) return 1;
      hipStreamSynchronize(&st);
      if (a != b) return 1;
    }
  }
  if (pinned != 0) return std::printf("%zu pinned bytes left\n", pinned), 1;
  std::printf("ok\n");
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("transfer")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (d / "main.cpp").write_text(MAIN)
    exe = d / "transfer"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", f"-I{d}", f"-I{CSRC}", str(d / "main.cpp"), "-o", str(exe)],
                   check=True)
    return exe


@pytest.mark.parametrize("what", ["plain", "known", "device", "memory", "unpinned"])
def test_threaded_copies(program, what):
    """Copies of several sizes up and down through one set of slots, which are
    no larger than the largest copy so far needs: as they are; of an array that the runtime knows; with a stream of another device
    than the current one; with no memory for one of the helper threads; and with
    none for the slots."""
    r = subprocess.run([str(program), what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout, r.stderr)
