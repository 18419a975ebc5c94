// How long the schedule tuners let a candidate run before they drop it.
#pragma once

namespace edl {

// A kernel's first launch loads its code and raises its LDS limit: up to a few
// hundred us of host time between the events, so that launch only drops a
// candidate that is slower than twice the best by more than this.
constexpr double kColdMs = 5.0;
// One launch between two events carries its launch latency, the mean of three
// hides most of it: kernels of a few us are all timed by three.
constexpr double kLatencyMs = 0.05;

// Mean ms of a launch of a candidate.  launch() queues one; clock(n) queues n and
// gives the ms they took.  A warm launch slower than twice the best so far ends
// the candidate (its time is returned, and is no new best).
template <typename Launch, typename Clock>
double candidate_ms(Launch launch, Clock clock, double best_ms) {
  if (best_ms > 1.0 && best_ms < 1e300) {
    const double first = clock(1);
    if (first > 2.0 * best_ms + kColdMs) return first;
  } else {
    launch();
  }
  const double one = clock(1);
  if (one > 2.0 * best_ms + kLatencyMs) return one;
  return clock(3) / 3;
}

}  // namespace edl
