// sd2d_xfer.hpp - copies between the caller's (pageable) arrays and the
// device.
//
// hipMemcpy of pageable memory moves the bytes through the runtime's own
// staging with one host thread, which also takes the page faults of a fresh
// output array.  Here the copy engine writes into (reads from) a ring of
// pinned slots while a few host threads move earlier (later) slots to (from)
// the caller's array.  To the host, 472 MB: 45 -> 12.5 ms (10.4 -> 37.7 GB/s;
// the link takes 57 GB/s into pinned memory), 29 MB: 1.75 -> 0.98 ms; to the
// device, 472 MB: 16.4 -> 12.3 ms.
//
// The ring (32 MiB) is one per process, allocated by the first large copy and
// freed with the last context.  A copy holds it alone: one that finds it
// taken (another context's, from another thread) or cannot get it uses plain
// hipMemcpyAsync.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>

namespace sd2d {

class HostRing {
 public:
  static constexpr int NSLOT_ = 16, LEAD = NSLOT_ / 2, MAXW = 8;
  static constexpr size_t SLOT = size_t(2) << 20;
  // To the host the runtime's copy is the faster one below 2.5 MiB (a state of 1.2
  // MiB: 127 against 147 us, 1.9 MiB: 160 against 202) and as fast up to 4 MiB (3.2:
  // 250 / 257, 4.0: 283 / 277, 4.8: 340 / 304, 7.8: 514 / 388); one host thread
  // more per 2 MiB.  To the device it is the faster one up to some tens of MB
  // (29 MB: 35 against 29 GB/s, 118 MB: 28 against 35).
  static constexpr size_t MIN_OUT = size_t(4) << 20, MIN_IN = size_t(64) << 20;

  static HostRing &get() {
    static HostRing r;
    return r;
  }
  // A context comes and goes without waiting for another's copy: the lock is held
  // only to take the ring and to give it back.  (A copy belongs to a context that
  // lives, so the ring has a user as long as it is taken.)
  void add_user() {
    std::lock_guard<std::mutex> lk(m_);
    ++users_;
  }
  void drop_user() {
    std::lock_guard<std::mutex> lk(m_);
    if (--users_ > 0) return;
    if (buf_) (void)hipHostFree(buf_);
    buf_ = nullptr;
  }

  // Copy `bytes` from the device to the host (out) or back, in stream order;
  // done only when the caller has synchronised the stream.
  hipError_t copy(hipStream_t st, void *host, void *dev, size_t bytes, bool out) {
    if (!pays(host, bytes, out) || !take()) return plain(st, host, dev, bytes, out);
    const hipError_t e = ring_copy(st, host, dev, bytes, out);
    std::lock_guard<std::mutex> lk(m_);
    busy_ = false;
    return e;
  }

 private:
  hipError_t ring_copy(hipStream_t st, void *host, void *dev, size_t bytes, bool out) {
    Job j;
    j.host = static_cast<char *>(host);
    j.ring = buf_;
    j.out = out;
    j.bytes = bytes;
    j.chunk = std::min(SLOT, std::max((bytes / 8 + 65535) & ~size_t(65535), size_t(262144)));
    j.n = (int)((bytes + j.chunk - 1) / j.chunk);
    hipEvent_t ev[NSLOT_] = {};
    hipError_t e = hipSuccess;
    const int ne = std::min(j.n, NSLOT_);
    for (int k = 0; k < ne && e == hipSuccess; ++k)
      e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
    std::thread th[MAXW];
    int nw = 0;
    if (e == hipSuccess) {
      const int want = std::min({MAXW, (int)std::max(1u, std::thread::hardware_concurrency() / 2),
                                 1 + (int)std::min<size_t>(MAXW, bytes / SLOT)});
      try {
        for (; nw < want; ++nw) th[nw] = std::thread([&j] { j.work(); });
      } catch (...) {   // no thread to be had: go on with those that started
      }
      e = nw ? drive(j, st, static_cast<char *>(dev), ev) : plain(st, host, dev, bytes, out);
    }
    {
      std::lock_guard<std::mutex> lk(j.m);
      j.stop = true;
    }
    j.cv.notify_all();
    for (int k = 0; k < nw; ++k) th[k].join();
    if (!out || e != hipSuccess) {   // no slot is reused before its copy has ended
      const hipError_t s = hipStreamSynchronize(st);
      if (e == hipSuccess) e = s;
    }
    for (hipEvent_t x : ev) if (x) (void)hipEventDestroy(x);
    return e;
  }

  struct Job {
    char *host, *ring;
    size_t bytes, chunk;
    int n;
    bool out;
    std::mutex m;
    std::condition_variable cv;
    int next = 0;            // next chunk a worker takes
    int open = 0;            // chunks below this may be moved by the host
    bool stop = false;
    int moved[NSLOT_] = {};  // last chunk + 1 the host moved through a slot

    size_t len(int k) const { return std::min(chunk, bytes - (size_t)k * chunk); }
    void move(int k) {
      char *h = host + (size_t)k * chunk, *r = ring + (size_t)(k % NSLOT_) * SLOT;
      if (out) std::memcpy(h, r, len(k));
      else std::memcpy(r, h, len(k));
    }
    void work() {
      std::unique_lock<std::mutex> lk(m);
      for (;;) {
        cv.wait(lk, [&] { return stop || next >= n || next < open; });
        if (next >= n || next >= open) return;   // all taken, or stopped
        const int k = next++;
        lk.unlock();
        move(k);
        lk.lock();
        moved[k % NSLOT_] = k + 1;
        cv.notify_all();
      }
    }
    void let(int upto) {
      {
        std::lock_guard<std::mutex> lk(m);
        open = upto;
      }
      cv.notify_all();
    }
    void wait_moved(int k) {
      std::unique_lock<std::mutex> lk(m);
      cv.wait(lk, [&] { return moved[k % NSLOT_] >= k + 1; });
    }
  };

  // The copy engine's side of a job.
  static hipError_t drive(Job &j, hipStream_t st, char *dev, hipEvent_t *ev) {
    hipError_t e = hipSuccess;
    auto dma = [&](int k) {
      char *r = j.ring + (size_t)(k % NSLOT_) * SLOT, *d = dev + (size_t)k * j.chunk;
      hipError_t x = j.out ? hipMemcpyAsync(r, d, j.len(k), hipMemcpyDeviceToHost, st)
                           : hipMemcpyAsync(d, r, j.len(k), hipMemcpyHostToDevice, st);
      return x != hipSuccess ? x : hipEventRecord(ev[k % NSLOT_], st);
    };
    if (j.out) {
      for (int k = 0; k < std::min(LEAD, j.n); ++k)
        if ((e = dma(k)) != hipSuccess) return e;
      for (int k = 0; k < j.n; ++k) {
        if ((e = hipEventSynchronize(ev[k % NSLOT_])) != hipSuccess) return e;
        j.let(k + 1);
        const int a = k + LEAD;   // its slot's last chunk was LEAD chunks ago
        if (a < j.n) {
          if (a >= NSLOT_) j.wait_moved(a - NSLOT_);
          if ((e = dma(a)) != hipSuccess) return e;
        }
      }
      for (int k = std::max(0, j.n - NSLOT_); k < j.n; ++k) j.wait_moved(k);
    } else {
      j.let(std::min(LEAD, j.n));
      for (int k = 0; k < j.n; ++k) {
        j.wait_moved(k);
        if ((e = dma(k)) != hipSuccess) return e;
        const int a = k + LEAD;   // chunk a's slot was last read by chunk a - NSLOT_
        if (a < j.n) {
          if (a >= NSLOT_ && (e = hipEventSynchronize(ev[a % NSLOT_])) != hipSuccess) return e;
          j.let(a + 1);
        }
      }
    }
    return e;
  }

  static hipError_t plain(hipStream_t st, void *host, void *dev, size_t bytes, bool out) {
    return out ? hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st)
               : hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st);
  }
  // Whether the ring moves these bytes faster than the runtime's copy.  The copy
  // engine reaches registered memory by itself: into pinned memory 472 MB take
  // 8.9 ms, through the ring 12.2 ms (8.1 MB: 0.20 and 0.38 ms).
  static bool pays(const void *host, size_t bytes, bool out) {
    if (bytes < (out ? MIN_OUT : MIN_IN)) return false;
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, host) == hipSuccess)
      return at.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();   // (some runtimes refuse pageable memory)
    return true;
  }

  // The ring for one copy, allocated by the first; false where another copy has it
  // or there is no memory for it.
  bool take() {
    std::lock_guard<std::mutex> lk(m_);
    if (busy_) return false;
    if (!buf_) {
      void *p = nullptr;
      if (hipHostMalloc(&p, NSLOT_ * SLOT, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
      buf_ = static_cast<char *>(p);
    }
    return busy_ = true;
  }

  std::mutex m_;          // users_, buf_, busy_
  int users_ = 0;
  bool busy_ = false;     // a copy has the ring
  char *buf_ = nullptr;
};

// A context's share in the ring.
struct RingUser {
  RingUser() { HostRing::get().add_user(); }
  ~RingUser() { HostRing::get().drop_user(); }
  RingUser(const RingUser &) = delete;
  RingUser &operator=(const RingUser &) = delete;
};

}  // namespace sd2d
