// galic_plan.h -- rules by which the FP32 path plans its response logs' memory and launches.  Host
// code without HIP (tests/test_log_plan.py runs it on the CPU).
#pragma once

#include <stddef.h>

#include <algorithm>

namespace galic {

// Whether a call keeps the log arena of `have` bytes that it finds.  It must hold `need`; then it
// is kept if it holds the call's orbits in one launch (`fit`), since a free and a new allocation of
// tens of GB cost more than most calls (0.4 s for 20 GB, 8 s for 130 GB), and a call that goes out
// in two launches lasts twice as long as its longest orbits.  A call that is `bounded`, because
// `want` is all that the memory allows or because a second arena takes its part, goes out in several
// launches whatever it does: it keeps an arena of half of what it wants, so that calls of different
// kinds in turn do not each take their own.
inline bool arena_kept(size_t have, size_t need, size_t want, size_t fit, bool bounded) {
  return have >= need && (have >= fit || (bounded && have >= want / 2));
}

// Orbits whose logs of `per_orbit` blocks fit `blocks`.  The lanes of a launch leave up to `chunk`
// blocks each unused: `slack` in all for a launch that fills the grid, and chunk an orbit and `group`
// lanes more for one that does not.  (Counted for the full grid alone, an arena below its slack,
// 8.4 GB, took its orbits one by one.)
inline double orbits_fit(double blocks, double slack, double chunk, double group, double per_orbit) {
  return std::max((blocks - slack) / per_orbit, (blocks - group * chunk) / (per_orbit + chunk));
}

// Orbits, from b0 on of m, whose logs (n[b] records each) make one commit of at most `most` records:
// one orbit at least.  Counted from the logs themselves: they are in the order of their expected
// length, so the first of m logs hold about twice the mean.
inline int commit_run(const int *n, int b0, int m, double most) {
  double records = 0;
  int b = b0;
  for(; b < m; b++) {
    records += n[b];
    if(b > b0 && records > most) break;
  }
  return b - b0;
}

// The step cap of the FP32 orbit kernel, whose counter is an int that is -1 at an orbit's start: one
// step more than the cap must be above it and not wrap to a negative count, which would start the
// orbit over for good.
inline long long fp32_step_cap(long long cap) { return std::min(cap, 0x7ffffffeLL); }

}  // namespace galic
