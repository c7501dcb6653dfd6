// PlanPoll (sched_policy.h) on the CPU, in the scheduler's loop: a poll's
// counters are read after the next poll's iterations are launched, those of the
// last one at once. A closed set of paths bounded by `bound` iterations whose last
// path ends after `life` of them finds its end and never runs past its bound; with
// bounds above kLaunchAhead an early end is noticed, and above kKnownAhead no more
// iterations run than without the bound. Prints "ok".
#include <algorithm>
#include <cstdio>

#include "sched_policy.h"

using namespace muonx;

// Iterations launched until the host knows that `life` of them were enough.
static uint64_t Run(uint64_t bound, uint64_t life, uint32_t per_poll) {
  uint64_t launched = 0, seen = 0;
  for (int steps = 0; seen < life && steps < 10000; ++steps) {
    const PollPlan p = PlanPoll(bound, launched, per_poll);
    const uint64_t before = launched;
    launched += p.iterations;
    seen = p.last ? launched : before;
  }
  return seen < life ? ~0ull : launched;
}

int main() {
  bool ok = true;
  for (uint64_t bound = 1; bound <= 60; ++bound)
    for (uint64_t life = 1; life <= bound; ++life)
      for (uint32_t per_poll : {1u, 2u, 3u, 4u, 8u, 16u, 100u}) {
        const uint64_t n = Run(bound, life, per_poll), plain = Run(0, life, per_poll);
        bool good = n >= life && n <= bound;
        if (bound <= kLaunchAhead) good = good && n == bound;
        else if (bound <= kKnownAhead) good = good && n <= std::max<uint64_t>(plain, life <= 8 ? 12 : bound);
        else good = good && n <= plain;
        if (!good) std::printf("bound %d life %d per poll %u: %d iterations, %d without the bound\n", int(bound), int(life), per_poll, int(n), int(plain));
        ok = ok && good;
      }
  // a bound that no launch reaches, and iterations past a bound (a set that was not done at it)
  ok = ok && PlanPoll(1ull << 31, 0, 2).iterations == 2 && !PlanPoll(1ull << 31, 0, 2).last;
  ok = ok && PlanPoll(5, 5, 2).iterations == 2 && !PlanPoll(5, 5, 2).last && !PlanPoll(5, 9, 2).last;
  std::puts(ok ? "ok" : "failed");
  return ok ? 0 : 1;
}
