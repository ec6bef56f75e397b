// Threads taking turns at a device's CUs: no moment holds more than all of
// them, a launch that needs every one comes through between small ones, one
// that gives up leaves the queue, and enter() returns within its limit.  With
// an argument only waits without a limit (ThreadSanitizer does not know the
// call that libstdc++'s timed waits make, and reports a double lock).
#include <assert.h>
#include <stdio.h>

#include <atomic>
#include <chrono>
#include <thread>
#include <vector>

#include "resident_gate.h"

using namespace smdp;
using Clock = std::chrono::steady_clock;

static double ms_since(Clock::time_point t) { return std::chrono::duration<double, std::milli>(Clock::now() - t).count(); }

int main(int argc, char**) {
  const bool timed = argc == 1;
  constexpr int kCus = 256;
  std::atomic<int> used{0}, most{0}, whole{0}, gave_up{0};
  auto work = [&](int units, int times, double wait_ms) {
    for (int i = 0; i < times; ++i) {
      ResidentShare share(3, units, kCus, wait_ms);
      if (!share.held()) {
        ++gave_up;
        continue;
      }
      const int now = used += std::min(units, kCus);
      for (int m = most; now > m && !most.compare_exchange_weak(m, now);) {
      }
      std::this_thread::sleep_for(std::chrono::microseconds(50));
      used -= std::min(units, kCus);
      if (units > kCus) ++whole;
    }
  };
  std::vector<std::thread> threads;
  for (int t = 0; t < 6; ++t) threads.emplace_back(work, 32 + 32 * t, 200, timed && t & 1 ? 0.2 : -1.0);
  threads.emplace_back(work, 1280, 100, -1.0);
  for (auto& t : threads) t.join();
  if (used != 0 || most > kCus || whole != 100) return 1;

  if (!timed) {
    printf("gate: ok\n");
    return 0;
  }
  // a second launch that does not fit waits for its limit and no longer ...
  ResidentShare first(5, 192, kCus);
  const auto t0 = Clock::now();
  ResidentShare second(5, 192, kCus, 20.0);
  if (!first.held() || second.held() || ms_since(t0) < 15.0) return 2;
  // ... one that fits beside the first goes in, also after one gave up ahead of it
  ResidentShare third(5, 64, kCus, 1000.0);
  if (!third.held()) return 3;
  // ... another device is not affected, and a release lets a waiting one in
  ResidentShare other(6, 256, kCus, 1000.0);
  if (!other.held()) return 4;
  std::atomic<bool> in{false};
  std::thread waiting([&] {
    ResidentShare s(5, 192, kCus);
    in = s.held();
  });
  std::this_thread::sleep_for(std::chrono::milliseconds(5));
  if (in) return 5;
  first.release();
  waiting.join();
  if (!in) return 6;
  printf("gate: ok, most %d, gave up %d\n", most.load(), gave_up.load());
  return 0;
}
