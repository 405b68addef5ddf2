// Host build of the count of compute units, for the CPU tests.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <memory>
#include <thread>

#include "hes_units.hpp"

using hes::ComputeUnits;

namespace {
// A launch on a thread of its own: comes at once, enters when it may, leaves
// when told to.
struct Launch {
  std::atomic<bool> in{false}, leave{false};
  std::thread t;
  Launch(int device, int need, bool waits)
      : t([=] {
          ComputeUnits u(device, 256, need, waits);
          in = true;
          while (!leave) std::this_thread::yield();
        }) {}
  ~Launch() {
    leave = true;
    t.join();
  }
  bool enters() {  // within a time that only a thread that may not enter exceeds
    for (int k = 0; k < 2000 && !in; ++k) std::this_thread::sleep_for(std::chrono::milliseconds(5));
    return in;
  }
  bool stays_out() {
    std::this_thread::sleep_for(std::chrono::milliseconds(100));
    return !in;
  }
};
int failures = 0;
void check(bool ok, const char* what) {
  if (!ok) {
    std::printf("failed: %s\n", what);
    ++failures;
  }
}
}  // namespace

int main() {
  {
    Launch a(0, 100, true), b(0, 156, true);
    check(a.enters() && b.enters(), "two teams that fit together");
    Launch other(1, 256, true);
    check(other.enters(), "another device");
    auto c = std::make_unique<Launch>(0, 1, true);
    check(c->stays_out(), "a team that does not fit beside them");
    auto d = std::make_unique<Launch>(0, 1, false);
    check(d->stays_out(), "a launch without waits that does not fit either");
    a.leave = true;
    check(c->enters() && d->enters(), "both once there is room");
  }
  {
    Launch a(0, 1000, false), b(0, 300, false);
    check(a.enters() && b.enters(), "launches without waits run beside one another");
    auto team = std::make_unique<Launch>(0, 2, true);
    check(team->stays_out(), "a team that finds the units held by launches without waits");
    auto late = std::make_unique<Launch>(0, 256, false);
    check(late->stays_out(), "a later launch that would pass the team over");
    a.leave = true;
    check(team->stays_out(), "a team beside the other one");
    b.leave = true;
    check(team->enters(), "a team once the units are free");
    check(late->stays_out(), "a launch of all units beside a team");
    team->leave = true;
    check(late->enters(), "the later launch, at last");
  }
  {
    Launch all(0, 256, true);
    check(all.enters(), "a team of all units");
    Launch none(0, 0, false);
    check(none.enters(), "a launch that holds no units");
  }
  return failures;
}
