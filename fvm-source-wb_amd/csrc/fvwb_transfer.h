// fvwb_transfer.h — copies of whole states between pageable host arrays and the
// device.
//
// The runtime's own copy to a pageable array goes through one thread and one
// staging buffer: 10.5 GB/s into fresh pages, 17.7 GB/s into touched ones, 29
// GB/s the other way (512 MB), where the link moves 57 GB/s.  Here a few host
// threads each take every T-th chunk through two pinned slots of their own, so
// the link, the page faults and the copies overlap: 41 GB/s into fresh pages and
// 46 GB/s the other way at 537 MB, 36 and 44 at 134 MB.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <thread>

namespace fvwb_xfer {

constexpr int THREADS = 4;                         // copies into fresh pages: 13, 41 and 48 GB/s with 1, 4 and 8
constexpr size_t SLOT = (size_t)4 << 20;           // at most, 32 MB of slots: with 1 and 2 MB 31 and 40 GB/s at 537 MB
// Where the threads' start costs what they save: to the host 0.56 ms either way
// at 8.4 MB, 0.76 against 1.06 at 15.7; to the device 0.58 against 0.48 at 15.7
// MB, 0.94 against 1.14 at 33.6.
constexpr size_t LEAST_DOWN = (size_t)8 << 20, LEAST_UP = (size_t)32 << 20;

// The pinned slots of one handle, made at its first large copy, as large as its
// largest copy needs (half of it, at most 32 MB) and kept until the handle goes.
// A slot's event marks its last transfer: every writer waits for it, on whichever
// stream it was.
// A handle pays for its slots once: where a process makes its first copies, a
// whole residual distribution program of 8.7 MB took 9.9 ms against 8.5 with the
// runtime's copy, one of 20.5 MB 11.6 against 11.0, one of 33.6 MB 6.0 against
// 13.3; later handles of the process 1.2 against 1.2, 2.4 against 3.3 and 6.0
// against 6.7.
struct Staging {
  char* slots = nullptr;
  size_t slot = 0;                                 // bytes of one
  hipEvent_t ev[2 * THREADS] = {};

  bool ready(size_t bytes) {
    if (slot >= bytes) return true;
    for (hipEvent_t& e : ev)
      if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return false;
    release();
    if (hipHostMalloc((void**)&slots, 2 * THREADS * bytes, hipHostMallocDefault) != hipSuccess) {
      slots = nullptr;
      return false;
    }
    slot = bytes;
    return true;
  }
  void release() {
    if (!slots) return;
    for (hipEvent_t e : ev) (void)hipEventSynchronize(e);
    (void)hipHostFree(slots);
    slots = nullptr;
    slot = 0;
  }
  Staging() = default;
  Staging(const Staging&) = delete;
  Staging& operator=(const Staging&) = delete;
  ~Staging() {
    release();
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
  }
};

// true if the runtime knows the array (pinned, managed or device memory): its
// own copy is then the fast one
inline bool known(const void* host) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, host) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

template <bool DOWN>
inline hipError_t copy(Staging& s, void* dst, const void* src, size_t bytes, hipStream_t st) {
  // about four chunks per thread or more, of 64 KB multiples
  const size_t chunk = std::min(SLOT, (bytes / (4 * THREADS) + 65535) / 65536 * 65536);
  // the threads and the events belong to the stream's device, which need not be
  // the caller's current one
  int mine = 0, dev = 0;
  bool staged = bytes >= (DOWN ? LEAST_DOWN : LEAST_UP) && !known(DOWN ? dst : src) &&
                hipGetDevice(&mine) == hipSuccess && hipStreamGetDevice(st, &dev) == hipSuccess;
  if (staged) {
    staged = hipSetDevice(dev) == hipSuccess && s.ready(chunk);
    if (!staged) (void)hipSetDevice(mine);
  }
  if (!staged) {
    (void)hipGetLastError();
    return hipMemcpyAsync(dst, src, bytes, DOWN ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, st);
  }
  const size_t n = (bytes + chunk - 1) / chunk;
  auto length = [&](size_t i) { return std::min(chunk, bytes - i * chunk); };
  hipError_t result[THREADS];
  auto work = [&](int t) {
    char* slot[2] = {s.slots + (size_t)(2 * t) * s.slot, s.slots + (size_t)(2 * t + 1) * s.slot};
    hipEvent_t ev[2] = {s.ev[2 * t], s.ev[2 * t + 1]};
    hipError_t e = hipSetDevice(dev);
    auto ok = [&](hipError_t r) {
      if (e == hipSuccess) e = r;
    };
    auto fetch = [&](size_t i, int k) {
      ok(hipMemcpyAsync(slot[k], (const char*)src + i * chunk, length(i), hipMemcpyDeviceToHost, st));
      ok(hipEventRecord(ev[k], st));
    };
    if (DOWN) {
      ok(hipEventSynchronize(ev[0]));
      ok(hipEventSynchronize(ev[1]));
      for (size_t i = t, k = 0; i < n && k < 2; i += THREADS, ++k) fetch(i, (int)k);
    }
    for (size_t i = t, k = 0; i < n && e == hipSuccess; i += THREADS, k ^= 1) {
      ok(hipEventSynchronize(ev[k]));
      if (e != hipSuccess) break;
      if (DOWN) {
        std::memcpy((char*)dst + i * chunk, slot[k], length(i));
        if (i + 2 * THREADS < n) fetch(i + 2 * THREADS, (int)k);
      } else {
        std::memcpy(slot[k], (const char*)src + i * chunk, length(i));
        ok(hipMemcpyAsync((char*)dst + i * chunk, slot[k], length(i), hipMemcpyHostToDevice, st));
        ok(hipEventRecord(ev[k], st));
      }
    }
    result[t] = e;
  };
  std::thread pool[THREADS];
  for (int t = 1; t < THREADS; ++t) {
    try {
      pool[t] = std::thread(work, t);
    } catch (...) {                                // no thread or no memory for one: its share is done below
    }
  }
  work(0);
  for (int t = 1; t < THREADS; ++t) {
    if (pool[t].joinable()) pool[t].join();
    else work(t);
  }
  (void)hipSetDevice(mine);
  for (hipError_t e : result)
    if (e != hipSuccess) return e;
  return hipSuccess;
}

// Both are ordered on `st` like hipMemcpyAsync.  A pageable host array of these
// sizes has been read, or filled, when they return; for any other the copy may
// still be under way, so the caller waits for the stream in either case.
inline hipError_t to_device(Staging& s, void* dst, const void* src, size_t bytes, hipStream_t st) {
  return copy<false>(s, dst, src, bytes, st);
}
inline hipError_t to_host(Staging& s, void* dst, const void* src, size_t bytes, hipStream_t st) {
  return copy<true>(s, dst, src, bytes, st);
}

}  // namespace fvwb_xfer
