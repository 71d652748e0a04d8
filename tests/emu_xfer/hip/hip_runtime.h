// CPU stand-ins for the HIP names that sd2d_xfer.hpp uses: a stream is a host
// thread that runs its operations in order, "device" memory is host memory,
// pinned memory is registered here, and every copy is counted by what its host
// side is.  Test infrastructure (tests/test_emu_xfer.py); the product library
// never sees this file.
#pragma once
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

#include <condition_variable>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <thread>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
struct hipPointerAttribute_t {
  hipMemoryType type;
};
constexpr unsigned hipHostMallocPortable = 1, hipEventDisableTiming = 2;

namespace fake {
struct Stream {
  std::mutex m;
  std::condition_variable cv;
  std::deque<std::function<void()>> q;
  bool held = false, end = false, idle = true;
  std::thread th{[this] {
    std::unique_lock<std::mutex> lk(m);
    for (;;) {
      cv.wait(lk, [&] { return (!held && !q.empty()) || (end && q.empty()); });
      if (q.empty()) return;
      auto f = q.front();
      q.pop_front();
      idle = false;
      lk.unlock();
      f();
      lk.lock();
      idle = true;
      cv.notify_all();
    }
  }};
  void add(std::function<void()> f) {
    {
      std::lock_guard<std::mutex> lk(m);
      q.push_back(std::move(f));
    }
    cv.notify_all();
  }
  void hold(bool on) {   // operations wait while the stream is held
    {
      std::lock_guard<std::mutex> lk(m);
      held = on;
    }
    cv.notify_all();
  }
  ~Stream() {
    {
      std::lock_guard<std::mutex> lk(m);
      end = true;
    }
    cv.notify_all();
    th.join();
  }
};
struct Event {
  std::mutex m;
  std::condition_variable cv;
  int recorded = 0, done = 0;
};
inline std::mutex mem_m;
inline std::map<char *, std::pair<size_t, hipMemoryType>> mem;   // registered ranges
inline size_t pinned_bytes = 0;                                   // allocated now
inline int direct_copies = 0, ring_copies = 0;                    // by the host side
inline hipMemoryType type_of(const void *p) {
  std::lock_guard<std::mutex> lk(mem_m);
  auto it = mem.upper_bound((char *)p);
  if (it == mem.begin()) return hipMemoryTypeUnregistered;
  --it;
  return (char *)p < it->first + it->second.first ? it->second.second : hipMemoryTypeUnregistered;
}
}  // namespace fake

using hipStream_t = fake::Stream *;
using hipEvent_t = fake::Event *;

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = malloc(n);
  std::lock_guard<std::mutex> lk(fake::mem_m);
  fake::mem[(char *)*p] = {n, hipMemoryTypeHost};
  fake::pinned_bytes += n;
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
  {
    std::lock_guard<std::mutex> lk(fake::mem_m);
    fake::pinned_bytes -= fake::mem[(char *)p].first;
    fake::mem.erase((char *)p);
  }
  free(p);
  return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  a->type = fake::type_of(p);
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
  const void *host = k == hipMemcpyDeviceToHost ? d : s;
  {
    std::lock_guard<std::mutex> lk(fake::mem_m);
    bool ring = false;   // the only pinned memory a test does not register by itself
    for (auto &r : fake::mem)
      if (r.second.second == hipMemoryTypeHost && (char *)host >= r.first &&
          (char *)host < r.first + r.second.first)
        ring = true;
    ++(ring ? fake::ring_copies : fake::direct_copies);
  }
  st->add([=] { memcpy(d, s, n); });
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t st) {
  std::unique_lock<std::mutex> lk(st->m);
  st->cv.wait(lk, [&] { return st->q.empty() && st->idle; });
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = new fake::Event;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
  int n;
  {
    std::lock_guard<std::mutex> lk(e->m);
    n = ++e->recorded;
  }
  st->add([=] {
    std::lock_guard<std::mutex> lk(e->m);
    e->done = n;
    e->cv.notify_all();
  });
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  std::unique_lock<std::mutex> lk(e->m);
  e->cv.wait(lk, [&] { return e->done >= e->recorded; });
  return hipSuccess;
}
