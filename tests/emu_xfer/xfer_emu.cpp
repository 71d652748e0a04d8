// xfer_emu.cpp - the host side of the state-sized copies (sd2d_xfer.hpp) on
// the CPU stand-ins of hip/hip_runtime.h, built with ThreadSanitizer by
// tests/test_emu_xfer.py.  Test infrastructure only.
//
//   xfer_emu data | contexts | pinned | small
#include "sd2d_xfer.hpp"

#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <future>
#include <random>
#include <string>
#include <vector>

using sd2d::HostRing;
using sd2d::RingUser;

#define CHECK(x)                                                             \
  do {                                                                       \
    if (!(x)) {                                                              \
      std::fprintf(stderr, "xfer_emu: %s (line %d)\n", #x, __LINE__);        \
      std::fflush(stderr);                                                   \
      std::_Exit(1);                                                         \
    }                                                                        \
  } while (0)

static std::vector<char> pattern(size_t n, unsigned seed) {
  std::vector<char> v(n);
  std::mt19937_64 r(seed);
  std::vector<uint64_t> w(4099);   // a period that no chunk size divides
  for (auto &x : w) x = r();
  for (size_t i = 0; i < n; i += 8 * w.size())
    std::memcpy(v.data() + i, w.data(), std::min(n - i, 8 * w.size()));
  return v;
}

// whole copies at the sizes where the path changes, to the host and back
static void data() {
  fake::Stream st;
  const size_t M = size_t(1) << 20;
  for (size_t n : {size_t(1000), M - 8, M, M + 8, 3 * M - 8, 3 * M, 4 * M - 8, 4 * M, 5 * M + 24,
                   17 * M + 8, 33 * M, 64 * M, 67 * M + 40}) {
    RingUser u;
    std::vector<char> dev = pattern(n, 1), host(n);
    CHECK(HostRing::get().copy(&st, host.data(), dev.data(), n, true) == hipSuccess);
    CHECK(hipStreamSynchronize(&st) == hipSuccess);
    CHECK(host == dev);
    host = pattern(n, 2);
    CHECK(HostRing::get().copy(&st, host.data(), dev.data(), n, false) == hipSuccess);
    CHECK(hipStreamSynchronize(&st) == hipSuccess);
    CHECK(host == dev);
  }
  CHECK(fake::pinned_bytes == 0);   // given back with the last context
}

// contexts come and go while another thread's copy waits for its stream, and a
// second copy goes another way
static void contexts() {
  fake::Stream st, st2;
  const size_t n = size_t(9) << 20;
  std::vector<char> dev = pattern(n, 3), host(n), dev2 = pattern(n, 4), host2(n);
  {
    RingUser u;
    st.hold(true);
    auto first = std::async(std::launch::async, [&] {
      return HostRing::get().copy(&st, host.data(), dev.data(), n, true);
    });
    for (;;) {   // until that copy has the ring
      {
        std::lock_guard<std::mutex> lk(fake::mem_m);
        if (fake::ring_copies > 0) break;
      }
      std::this_thread::yield();
    }
    auto come_and_go = std::async(std::launch::async, [] {
      for (int i = 0; i < 3; ++i) RingUser other;
    });
    CHECK(come_and_go.wait_for(std::chrono::seconds(20)) == std::future_status::ready);
    CHECK(HostRing::get().copy(&st2, host2.data(), dev2.data(), n, true) == hipSuccess);
    CHECK(hipStreamSynchronize(&st2) == hipSuccess);
    CHECK(host2 == dev2);
    st.hold(false);
    CHECK(first.get() == hipSuccess);
    CHECK(hipStreamSynchronize(&st) == hipSuccess);
    CHECK(host == dev);
    CHECK(fake::pinned_bytes > 0);
  }
  CHECK(fake::pinned_bytes == 0);
}

// an array the copy engine reaches by itself is copied in one piece
static void pinned() {
  fake::Stream st;
  RingUser u;
  const size_t n = size_t(70) << 20;
  std::vector<char> dev = pattern(n, 5);
  void *p = nullptr;
  CHECK(hipHostMalloc(&p, n, 0) == hipSuccess);
  for (bool out : {true, false}) {
    fake::ring_copies = 0;   // (counts every copy whose host side is pinned)
    CHECK(HostRing::get().copy(&st, p, dev.data(), n, out) == hipSuccess);
    CHECK(hipStreamSynchronize(&st) == hipSuccess);
    CHECK(fake::ring_copies == 1 && fake::direct_copies == 0);
    CHECK(std::memcmp(p, dev.data(), n) == 0);
  }
  CHECK(fake::pinned_bytes == n);
  CHECK(hipHostFree(p) == hipSuccess);
}

// below the sizes where the ring is the faster way, a copy is one of the runtime's
static void small() {
  fake::Stream st;
  RingUser u;
  const size_t M = size_t(1) << 20;
  for (size_t n : {M, 2 * M, 3 * M + 8, 4 * M - 8}) {
    std::vector<char> dev = pattern(n, 6), host(n);
    for (bool out : {true, false}) {
      fake::direct_copies = 0;
      CHECK(HostRing::get().copy(&st, host.data(), dev.data(), n, out) == hipSuccess);
      CHECK(hipStreamSynchronize(&st) == hipSuccess);
      CHECK(fake::direct_copies == 1 && fake::ring_copies == 0);
    }
  }
  CHECK(fake::pinned_bytes == 0);
}

int main(int argc, char **argv) {
  const std::string job = argc > 1 ? argv[1] : "";
  if (job == "data") data();
  else if (job == "contexts") contexts();
  else if (job == "pinned") pinned();
  else if (job == "small") small();
  else return 2;
  return 0;
}
