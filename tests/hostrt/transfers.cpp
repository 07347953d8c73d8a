// One call of the transfers a line of arguments, on the host runtime beside
// this file; prints what the call did.
#include <atomic>
#include <cstdio>
#include <new>
#include <string>
#include <vector>

#include "rhy_transfer.hip"

// The allocation that fails: counted down by every one while at or above 0.
static std::atomic<int> g_fail_at{-1};
void* operator new(size_t n) {
  if (g_fail_at.load() >= 0 && g_fail_at.fetch_sub(1) == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace {

// n values there and back, checked; true if both were right.
bool round_trip(size_t n, bool as_double, bool up, bool down, FakeStream* s) {
  const size_t esz = as_double ? 4 : 8;
  std::vector<unsigned char> dev(n * esz);
  std::vector<double> host(n), back(n);
  for (size_t i = 0; i < n; ++i) host[i] = (double)(i % 4099) * 0.25;
  bool ok = true;
  if (up) {
    const rhy::HostSpan span = {dev.data(), host.data(), n};
    ok = rhy::copy_spans(s, &span, 1, esz, as_double, false) == hipSuccess;
  }
  for (size_t i = 0; i < n; ++i) {
    if (as_double) {
      float& f = reinterpret_cast<float*>(dev.data())[i];
      if (up) ok = ok && f == (float)host[i];
      f = (float)host[i];
    } else {
      double& d = reinterpret_cast<double*>(dev.data())[i];
      if (up) ok = ok && d == host[i];
      d = host[i];
    }
  }
  if (down) {
    const rhy::HostSpan span = {dev.data(), back.data(), n};
    ok = ok && rhy::copy_spans(s, &span, 1, esz, as_double, true) == hipSuccess && back == host;
  }
  return ok;
}

}  // namespace

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  FakeStream s{0};
  bool ok = false;
  if (what == "route") {  // route KIB mixed|same up|down: a copy by a long-lived object
    const bool mixed = std::string(argv[3]) == "mixed", up = std::string(argv[4]) == "up";
    const size_t n = std::stoul(argv[2]) * 1024 / (mixed ? 4 : 8);
    rhy::transfer_user_add();
    ok = true;
    for (size_t moved = 0; ok && moved < (size_t)128 << 20; moved += n * (mixed ? 4 : 8)) {
      hostrt::copies = 0;
      ok = round_trip(n, mixed, up, !up, &s);
    }
    std::printf("copies %d ", hostrt::copies);
    rhy::transfer_user_drop();
  }
  if (what == "short") {  // objects that copy 12 MiB to the host and go
    ok = true;
    for (int i = 0; i < 20 && ok; ++i) {
      rhy::transfer_user_add();
      ok = round_trip((size_t)3 << 19, false, false, true, &s);
      rhy::transfer_user_drop();
    }
    std::printf("asked %d ", hostrt::pinned_calls);
  }
  if (what == "long") {  // one that makes the same copies
    ok = true;
    rhy::transfer_user_add();
    for (int i = 0; i < 20 && ok; ++i) ok = round_trip((size_t)3 << 19, false, false, true, &s);
    std::printf("asked %d held %d ", hostrt::pinned_calls, hostrt::pinned_bytes > 0);
    rhy::transfer_user_drop();
  }
  if (what == "refused") {  // no pinned memory to be had
    hostrt::refuse_pinned = ok = true;
    rhy::transfer_user_add();
    for (int i = 0; i < 5 && ok; ++i) ok = round_trip((size_t)8 << 20, false, true, true, &s);
    std::printf("asked %d copies %d ", hostrt::pinned_calls, hostrt::copies);
    rhy::transfer_user_drop();
  }
  if (what == "wait") {  // a caller that waits for the stream itself
    std::vector<double> dev(1000), host(1000, 1.5);
    const rhy::HostSpan span = {dev.data(), host.data(), host.size()};
    ok = rhy::copy_spans(&s, &span, 1, 8, false, false, false) == hipSuccess;
    std::printf("unwaited %d ", hostrt::waits);
    ok = ok && rhy::copy_spans(&s, &span, 1, 8, false, false) == hipSuccess;
    std::printf("waited %d ", hostrt::waits);
  }
  if (what == "pinned") {  // caller memory the runtime knows
    std::vector<double> dev((size_t)8 << 20), host((size_t)8 << 20, 1.5);
    hostrt::pinned_lo = host.data();
    hostrt::pinned_hi = host.data() + host.size();
    const rhy::HostSpan span = {dev.data(), host.data(), host.size()};
    rhy::transfer_user_add();
    ok = rhy::copy_spans(&s, &span, 1, 8, false, false) == hipSuccess && dev == host &&
         rhy::copy_spans(&s, &span, 1, 8, false, true) == hipSuccess;
    rhy::transfer_user_drop();
    std::printf("copies %d ", hostrt::copies);
  }
  if (what == "device") {  // a box of device 0 while the caller's is device 1
    hostrt::device = 1;
    rhy::transfer_user_add();
    ok = round_trip((size_t)8 << 20, false, true, true, &s) && hostrt::copies > 2;  // 64 MiB
    rhy::transfer_user_drop();
    std::printf("current %d ", hostrt::device);
  }
  if (what == "memory") {  // every allocation of a first copy fails in turn
    const size_t n = (size_t)8 << 20;
    std::vector<double> dev(n), host(n);
    ok = true;
    for (int at = 0; at < 40 && ok; ++at) {
      for (size_t i = 0; i < n; i += 997) host[i] = (double)at + 1.0;
      const rhy::HostSpan span = {dev.data(), host.data(), n};
      rhy::transfer_user_add();
      g_fail_at = at;
      ok = rhy::copy_spans(&s, &span, 1, 8, false, false) == hipSuccess;
      g_fail_at = -1;
      ok = ok && dev == host;
      rhy::transfer_user_drop();
    }
  }
  std::printf("ok %d events %d pinned %zu\n", ok, hostrt::events, hostrt::pinned_bytes);
  return ok ? 0 : 1;
}
