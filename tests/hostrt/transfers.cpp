// One call of the transfers a line of arguments, on the host runtime beside
// this file; prints what the call did.
#include <cstdio>
#include <string>
#include <vector>

#include "rhy_transfer.hip"

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
    ok = round_trip((size_t)8 << 20, false, true, true, &s) && hostrt::copies > 2;
    rhy::transfer_user_drop();
    std::printf("current %d ", hostrt::device);
  }
  std::printf("ok %d events %d pinned %zu\n", ok, hostrt::events, hostrt::pinned_bytes);
  return ok ? 0 : 1;
}
