// A wait of more polls than 32 bits count must still end: QuietTimeout (csrc/plugin/trace.h) against a clock that the
// polls themselves move, at 25 to 40 ns a poll.
#include <cstdio>

#include "trace.h"

static bool ends_in_time(double poll_s, double timeout_s) {
  tcpx::QuietTimeout quiet;
  double now = 1000.0;
  for (unsigned long long polls = 1; polls < 6000000000ull; ++polls) {
    now += poll_s;
    if (!quiet.expired(timeout_s, [&] { return now; })) continue;
    const double waited = now - 1000.0, slack = 2 * tcpx::QuietTimeout::kPollsPerLook * poll_s + 1e-3;
    std::printf("poll %.0f ns, time-out %.3f s: ended after %llu polls, %.3f s\n", poll_s * 1e9, timeout_s, polls, waited);
    return waited >= timeout_s && waited <= timeout_s + slack;
  }
  std::printf("poll %.0f ns, time-out %.3f s: never ended\n", poll_s * 1e9, timeout_s);
  return false;
}

int main() {
  if (!ends_in_time(30e-9, 0.05) || !ends_in_time(40e-9, 180.0)) return 1;  // (180 s: 4.5e9 polls)
  tcpx::QuietTimeout quiet;  // a poll that finds something starts the wait again
  double now = 0;
  for (int i = 0; i < 1000000; ++i) {
    now += 1e-3;
    if (i % 500 == 499) quiet.reset();
    if (quiet.expired(1.0, [&] { return now; })) return 1;
  }
  std::puts("quiet time-out ok");
  return 0;
}
