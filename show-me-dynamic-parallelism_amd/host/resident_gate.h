// Host-only: turns at a device's CUs for launches whose workgroups wait for one
// another.
//
// Such a launch needs all its workgroups resident at once.  It is sized for an
// idle device, but two contexts (one per host thread) may have one each in
// flight: 192 + 192 workgroups of a CU each on 256 CUs can be dispatched in
// turn until neither launch is whole, and both then poll their barriers until
// they give up, about a second later, for solves of 0.3 ms.  So every such
// launch first takes as many CUs as it has workgroups (at most all of them),
// and holds them until it has completed.  A workgroup keeps at most one CU from
// another launch, wherever it is placed, so launches that hold no more than all
// CUs together are whole at once.  Launches without barriers take no part: they
// end by themselves.  Other processes on the device are not seen here; against
// them the bounded barriers remain.
//
// First come, first served, so a launch that needs every CU is not passed over
// by small ones for ever.
#pragma once
#include <algorithm>
#include <chrono>
#include <condition_variable>
#include <list>
#include <mutex>

namespace smdp {

class ResidentGate {
 public:
  // Waits for `cus` of the device's `total` CUs, for at most wait_ms
  // milliseconds (below 0: without limit); false when they were not free by
  // then.
  bool enter(int cus, int total, double wait_ms = -1.0) {
    std::unique_lock<std::mutex> lock(mutex_);
    const auto me = queue_.insert(queue_.end(), 0);
    auto mine = [&] { return queue_.begin() == me && used_ + cus <= total; };
    bool ok = true;
    if (wait_ms < 0) changed_.wait(lock, mine);
    else ok = changed_.wait_for(lock, std::chrono::duration<double, std::milli>(wait_ms), mine);
    queue_.erase(me);
    if (ok) used_ += cus;
    changed_.notify_all();  // the next in the queue may fit beside this one
    return ok;
  }
  void leave(int cus) {
    std::lock_guard<std::mutex> lock(mutex_);
    used_ -= cus;
    changed_.notify_all();
  }

 private:
  std::mutex mutex_;
  std::condition_variable changed_;
  std::list<int> queue_;
  int used_ = 0;
};

// The gate of a device (devices beyond the table share one, which only makes
// them wait for each other).
inline ResidentGate& resident_gate(int device) {
  static ResidentGate gates[64];
  return gates[device & 63];
}

// The CUs of one launch of `workgroups` workgroups, from construction until
// release() or the end of the scope: after the host has waited for the launch.
class ResidentShare {
 public:
  ResidentShare(int device, int workgroups, int total, double wait_ms = -1.0)
      : gate_(resident_gate(device)), cus_(std::max(1, std::min(workgroups, total))) {
    held_ = gate_.enter(cus_, std::max(1, total), wait_ms);
  }
  ~ResidentShare() { release(); }
  ResidentShare(const ResidentShare&) = delete;
  ResidentShare& operator=(const ResidentShare&) = delete;
  bool held() const { return held_; }
  void release() {
    if (held_) gate_.leave(cus_);
    held_ = false;
  }

 private:
  ResidentGate& gate_;
  const int cus_;
  bool held_ = false;
};

}  // namespace smdp
