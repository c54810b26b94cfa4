// lusgs_plan.h — the schedule of the LU-SGS sweeps in plain C++: the order of the
// patches, the places of what they hand over, and their waits (the library and its
// sweep kernel run it, a CPU test compiles it).
#pragma once

#include <algorithm>
#include <cstddef>
#include <vector>

#ifdef __HIP__
#define CFX_HD __host__ __device__
#else
#define CFX_HD
#endif

namespace cfx {

// LU-SGS sweeps: patches of kLuP x kLuP columns along i; the patch (J, K) of a
// block, in the order in which wavefronts take them (any patch behind (J-1, K)
// and (J, K-1)).
constexpr int kLuP = 4;
struct LuPatch {
  int blk, J, K;
};

// The order over all blocks of my[b] x mz[b] columns, by J + K, and behind it each
// block's own list (index 0); off: where the lists of the blocks begin, and the end.
inline void lu_plan(const std::vector<int> &my, const std::vector<int> &mz, std::vector<LuPatch> &order,
                    std::vector<int> &off) {
  std::vector<LuPatch> own;
  std::vector<int> count;
  order.clear();
  for (size_t b = 0; b < my.size(); ++b) {
    const int nj = (my[b] + kLuP - 1) / kLuP, nk = (mz[b] + kLuP - 1) / kLuP;
    for (int d = 0; d <= nj + nk - 2; ++d)
      for (int K = std::max(0, d - nj + 1); K <= std::min(d, nk - 1); ++K) {
        order.push_back(LuPatch{(int)b, d - K, K});
        own.push_back(LuPatch{0, d - K, K});
      }
    count.push_back(nj * nk);
  }
  std::stable_sort(order.begin(), order.end(),
                   [](const LuPatch &x, const LuPatch &y) { return x.J + x.K < y.J + y.K; });
  off.assign(1, (int)order.size());
  for (int c : count) off.push_back(off.back() + c);
  order.insert(order.end(), own.begin(), own.end());
}

// A third of the species, and the places of a cell's variables: (rho, rho V, E)
// and three groups of species.
CFX_HD constexpr int lu_third(int ns) { return (ns + 2) / 3; }
CFX_HD constexpr int lu_places(int ns) { return 5 + 3 * lu_third(ns); }

// What a patch hands to the next one along j, and along k, is a record per step:
// the terms of its last columns, [variable of a group][group][column], so that a
// step's values are a few whole lines.  Group 0 alone has variables from N3 on.
CFX_HD constexpr int lu_record(int ns) { return kLuP * lu_places(ns); }
CFX_HD constexpr int lu_place(int ns, int q) {
  return q < lu_third(ns) ? 4 * kLuP * q : (3 * lu_third(ns) + q) * kLuP;
}
CFX_HD inline int lu_steps(int mx, int my, int mz) {
  return mx + (my < kLuP ? my : kLuP) + (mz < kLuP ? mz : kLuP) - 2;
}
// first value of a lane of a group in the record of a patch (K nj + J) at a step
CFX_HD inline long long lu_at(int ns, int steps, long long patch, int step, int group, int column) {
  return (patch * steps + step) * lu_record(ns) + kLuP * group + column;
}
// where the records for the patches after them along k begin, and the size of both
// kinds (either only where there are several patches)
CFX_HD inline long long lu_along_k(int ns, int mx, int my, int mz) {
  const long long nj = (my + kLuP - 1) / kLuP, nk = (mz + kLuP - 1) / kLuP;
  return nj > 1 ? nj * nk * lu_steps(mx, my, mz) * lu_record(ns) : 0;
}
CFX_HD inline long long lu_hand_over(const int m[3], int ns) {
  const long long nj = (m[1] + kLuP - 1) / kLuP, nk = (m[2] + kLuP - 1) / kLuP;
  return lu_along_k(ns, m[0], m[1], m[2]) + (nk > 1 ? nj * nk * lu_steps(m[0], m[1], m[2]) * lu_record(ns) : 0);
}
// At step s a column (jl, kl) of a patch is at the cell i = s - jl - kl, if that is
// one; a cell that the patch before updates in its step s + kLuP - 1 is the upstream
// neighbour of the one here.
CFX_HD inline bool lu_active(int mx, int jl, int kl, int s) { return s >= jl + kl && s < mx + jl + kl; }
constexpr int kLuAhead = kLuP - 1;

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
