// wait_guard.h -- when an object's solves may run in kernels whose workgroups
// wait for each other.
#pragma once

#include <algorithm>

namespace hg {

// Such a kernel needs its workgroups to run at the same time.  Where other
// processes or streams keep some of them off the GPU, its waits end after a
// number of polls and the solve is run again by kernels that do not wait.  That
// bound is long against a solve (0.1 s and more), so after a solve that gave up
// the next 16 do not try; twice as many after each further one in a row, up to
// 1024.
class WaitGuard {
 public:
  // May the next solve wait?
  bool Try() {
    if (skip_ == 0) return true;
    --skip_;
    return false;
  }
  void Finished() { next_ = kFirst; }
  void GaveUp() {
    ++give_ups_;
    skip_ = next_;
    next_ = std::min(2 * next_, kMost);
  }
  // The bound in polls (negative: each kernel's own); solves wait again.
  void SetPolls(int polls) {
    polls_ = polls;
    skip_ = 0;
    next_ = kFirst;
  }
  int Polls(int own) const { return polls_ < 0 ? own : polls_; }
  long give_ups() const { return give_ups_; }

 private:
  static constexpr int kFirst = 16, kMost = 1024;
  int polls_ = -1, skip_ = 0, next_ = kFirst;
  long give_ups_ = 0;
};

}  // namespace hg
