// Whose turn it is to hold compute units of a device (cg_resident.hip).
#pragma once

#include <condition_variable>
#include <mutex>

namespace alien_hip {

// The launches of the process whose workgroups wait for one another, on one device: together they hold no more
// compute units than it has, so that every workgroup of each runs (two that each hold half of what the other one still
// needs would wait for good). In the order in which they come, so that none is passed by for ever.
struct ResidentGate {
  std::mutex m;
  std::condition_variable cv;
  unsigned next = 0, serving = 0;
  int used = 0;
};

// A share of `blocks` compute units of `cus`, from here to the end of the scope; none (and no wait) for 0 blocks.
class ResidentTurn {
 public:
  ResidentTurn(ResidentGate& gate, int blocks, int cus) : g(gate), n(blocks) {
    if (n == 0) return;
    std::unique_lock<std::mutex> l(g.m);
    const unsigned t = g.next++;
    g.cv.wait(l, [&] { return t == g.serving && (g.used == 0 || g.used + n <= cus); });
    ++g.serving;
    g.used += n;
    g.cv.notify_all();
  }
  ~ResidentTurn() {
    if (n == 0) return;
    const std::lock_guard<std::mutex> l(g.m);
    g.used -= n;
    g.cv.notify_all();
  }
  ResidentTurn(const ResidentTurn&) = delete;
  ResidentTurn& operator=(const ResidentTurn&) = delete;

 private:
  ResidentGate& g;
  int n;
};

ResidentGate& resident_gate(int device);

} // namespace alien_hip
