// lusgs_plan.h — the waits of the LU-SGS sweeps, in plain C++ (the sweep kernel
// runs it, a CPU test compiles it).
#pragma once

#ifdef __HIP__
#define CFX_HD __host__ __device__
#else
#define CFX_HD
#endif

namespace cfx {

// A patch waits until the terms that it needs are there: while missing(), poll()
// loads them again.  A wait beyond `limit` of clock() is given up, which the order
// of the patches does not allow to happen: give_up() then records the error and
// raises the sweep's abort word, and a wait that finds the word raised
// (given_up(), every kLuPolls polls) ends too, so that the sweep comes to its end.
// The word belongs to one sweep and is cleared before the next: what was reported
// earlier must not cut short the waits of a later sweep, whose patches are running.
// Returns whether the terms are there.
constexpr int kLuPolls = 256;
template <class Missing, class Poll, class Clock, class GiveUp, class GivenUp>
CFX_HD inline bool lu_wait(Missing missing, Poll poll, Clock clock, long long limit, GiveUp give_up, GivenUp given_up) {
  if (!missing()) return true;
  const long long until = clock() + limit;
  for (int spin = 1; missing(); ++spin) {
    poll();
    if (spin % kLuPolls) continue;
    if (clock() > until) give_up();
    if (given_up()) return false;
  }
  return true;
}

}  // namespace cfx
