// hes_units.hpp -- which one-launch time loops may be on a device at once.
#pragma once
#include <condition_variable>
#include <mutex>

namespace hes {

// The compute units of a launch that holds them for many time steps.  Where its
// workgroups wait for one another (`waits`) it may only run beside other such
// launches if all fit: each could hold units that the other's missing workgroups
// need, and workgroups that start late would use up the time that the others
// wait.  Launches without waits end by themselves and only keep those with
// waits out.  All enter in the order in which they came, so none is passed over
// for ever.  Held from before the launch until its stream has been waited for;
// a launch that needs none is not counted.
class ComputeUnits {
 public:
  ComputeUnits(int device, int total, int need, bool waits)
      : s_(state(device)), need_(need < total ? need : total), waits_(waits) {
    if (need_ == 0) return;
    std::unique_lock<std::mutex> lock(s_.mutex);
    const unsigned long long turn = s_.came++;
    s_.cv.wait(lock, [&] {
      return s_.turn == turn &&
             (s_.used + need_ <= total || (waits_ ? s_.used == 0 : s_.waiting == 0));
    });
    ++s_.turn;
    s_.used += need_;
    s_.waiting += waits_;
    s_.cv.notify_all();
  }
  ~ComputeUnits() {
    if (need_ == 0) return;
    std::lock_guard<std::mutex> lock(s_.mutex);
    s_.used -= need_;
    s_.waiting -= waits_;
    s_.cv.notify_all();
  }
  ComputeUnits(const ComputeUnits&) = delete;
  ComputeUnits& operator=(const ComputeUnits&) = delete;

 private:
  struct State {
    std::mutex mutex;
    std::condition_variable cv;
    unsigned long long came = 0, turn = 0;  // launches that came; the next to enter
    int used = 0, waiting = 0;              // units held; launches with waits among the holders
  };
  static State& state(int device) {  // devices that share one only wait longer
    static State s[64];
    return s[device & 63];
  }
  State& s_;
  int need_;
  bool waits_;
};

}  // namespace hes
