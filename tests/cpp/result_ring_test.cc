// Checks on the CPU that no two requests in flight on a slot share a result
// entry, whichever requests failed before they got to it.  Exit status 0 on
// success.
#include <cstdio>
#include <deque>
#include <random>

#include "result_ring.h"

namespace {

template <uint32_t kDepth>
int run(uint32_t seed, double failing) {
  std::mt19937 rng(seed);
  std::uniform_real_distribution<double> u(0.0, 1.0);
  lbvh::ResultRing<kDepth> ring;
  uint32_t words[kDepth] = {};      // what the epilogues wrote
  std::deque<uint32_t> in_flight;   // serials, oldest first
  size_t written = 0;               // of in_flight: their epilogues ran
  for (int step = 0; step < 20000; ++step) {
    if (u(rng) < 0.4 && in_flight.size() < kDepth) {
      const int want = u(rng) < failing ? 4 : 0;
      uint32_t serial = 0;
      if (ring.admit(&serial, [&] { return want; }) != want) return 1;
      if (want == 0) in_flight.push_back(serial);
    }
    if (u(rng) < 0.4 && written < in_flight.size()) {  // in stream order
      const uint32_t s = in_flight[written++];
      words[ring.entry(s)] = s;
    }
    // every epilogue that ran shows, none that did not
    for (size_t k = 0; k < in_flight.size(); ++k) {
      const bool done = words[ring.entry(in_flight[k])] == in_flight[k];
      if (done != (k < written)) {
        std::fprintf(stderr, "step %d: request %zu of %zu in flight is %s\n",
                     step, k, in_flight.size(), done ? "done" : "lost");
        return 1;
      }
    }
    if (u(rng) < 0.4 && written > 0) {
      in_flight.pop_front();
      --written;
    }
  }
  return 0;
}

}  // namespace

int main() {
  for (uint32_t seed = 1; seed <= 5; ++seed)
    for (double failing : {0.0, 0.1, 0.9})
      if (run<1>(seed, failing) || run<2>(seed, failing) || run<4>(seed, failing))
        return 1;
  std::puts("ok");
  return 0;
}
