// How long the schedule tuners let a candidate run before they drop it.
#pragma once

#include <algorithm>

namespace edl {

// A kernel's first launch loads its code and raises its LDS limit, host time
// between the events: a first launch drops a candidate only beyond this much.
constexpr double kColdMs = 0.5;
// A single launch carries its launch latency, most of which the mean of three hides.
constexpr double kLatencyMs = 0.05;
// Below this a candidate's launches cost less than the waits that dropping it
// early would take.
constexpr double kSmallMs = 0.2;

// Mean ms of a launch of a candidate.  launch() queues one; clock(n) queues n and
// gives the ms they took.  Launches of kSmallMs and more drop a candidate as soon
// as a warm one is a tenth slower than the best so far (single launches of these
// sizes repeat within 3 %): its time is returned, and is no new best.  Tuning on
// the 4x4 sector in fp64: the operator 8.2 -> 3.9 s (there a cold first launch
// slower than twice the best dropped a candidate), a chain's shapes 3.1 -> 1.6 s
// (there every candidate ran four launches).
template <typename Launch, typename Clock>
double candidate_ms(Launch launch, Clock clock, double best_ms) {
  if (best_ms >= kSmallMs && best_ms < 1e300) {
    const double limit = best_ms + std::max(0.1 * best_ms, kLatencyMs);
    const double first = clock(1);
    if (first > limit + kColdMs) return first;
    if (first > limit) {
      const double one = clock(1);
      if (one > limit) return one;
    }
  } else {
    launch();
  }
  return clock(3) / 3;
}

}  // namespace edl
