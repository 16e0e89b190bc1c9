// Checks of the turns at a device's compute units (kernels/resident_turn.h), run by tests/test_resident_turn.py.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>

#include "kernels/resident_turn.h"

using namespace alien_hip;

static int failed = 0;
static void check(bool c, const char* what) {
  if (!c) std::printf("FAILED: %s\n", what);
  failed += !c;
}
static void pause_ms(int ms) { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); }

int main() {
  ResidentGate g;
  {
    const ResidentTurn a(g, 100, 256), b(g, 156, 256); // together
    const ResidentTurn none(g, 0, 256);                // a launch that waits for no other
    check(g.used == 256, "two launches that fit hold their shares at once");
  }
  check(g.used == 0, "shares are given back");
  {
    // one that does not fit waits, and one behind it that would fit does not pass it by
    std::atomic<int> order{0}, big{0}, small{0};
    std::thread t1, t2;
    {
      const ResidentTurn a(g, 100, 256);
      t1 = std::thread([&] {
        const ResidentTurn b(g, 200, 256);
        big = ++order;
      });
      while (true) { // until it has taken its number
        const std::lock_guard<std::mutex> l(g.m);
        if (g.next - g.serving == 1) break;
      }
      t2 = std::thread([&] {
        const ResidentTurn c(g, 100, 256);
        small = ++order;
      });
      while (true) {
        const std::lock_guard<std::mutex> l(g.m);
        if (g.next - g.serving == 2) break;
      }
      pause_ms(20);
      check(order == 0, "what does not fit waits, and what comes after it");
    }
    t1.join();
    t2.join();
    check(big == 1 && small == 2, "in the order in which they came");
  }
  {
    std::atomic<int> held{0}, most{0}, turns{0};
    std::vector<std::thread> ts;
    for (int k = 0; k < 8; ++k)
      ts.emplace_back([&, k] {
        for (int i = 0; i < 300; ++i) {
          const int n = 1 + (i * 37 + k * 101) % 256;
          const ResidentTurn t(g, n, 256);
          const int now = held += n;
          for (int m = most; now > m && !most.compare_exchange_weak(m, now);) {
          }
          held -= n;
          ++turns;
        }
      });
    for (auto& t : ts) t.join();
    check(turns == 8 * 300 && most <= 256 && g.used == 0, "never more than the device has");
  }
  if (!failed) std::printf("ok\n");
  return failed != 0;
}
