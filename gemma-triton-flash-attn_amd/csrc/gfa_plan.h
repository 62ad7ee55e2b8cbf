// How a split dK/dV grid is divided into workgroups: host code without allocations, exceptions or
// library calls.
#pragma once
#include <stdint.h>

#include <algorithm>

#include "gfa_params.h"

namespace gfa {

// Split counts of a dK/dV grid whose key blocks are split (q_splits > 1), and its workgroups.
//
// q_splits equal chunks per key block keep every CU busy, but under causal masking the late blocks
// need fewer, and every split costs fp32 partial rows: 64 keys x 512 columns of dK and dV are 256 KB
// written and read again, so that on small grids the partials took a third of the stage. Chunks
// of one length over the whole grid need half the splits, and one round of them ends together.
// Which is shorter is a matter of rounding (a few chunks past one round cost a second one), so
// the candidates are run through a list schedule of their workgroups: equal splits, and the
// shortest common chunk that gives at most 1, 1.5 or 2 rounds. Costs in iterations (one query tile
// of one head, 2 us at D = 512): a workgroup's prologue and epilogue take about 8, a split's
// partials 0.03 of the whole GPU. delta + dK/dV + reduction, us, before and after: D=256 8:4
// soft-capped N=1709 87.9 -> 66, N=3000 173 -> 132; 16:8 N=800 71 -> 47, N=1709 151 -> 90; D=512
// 16:2 N=2048 218 -> 189; D=64 2x16:16 N=2001 50.5 -> 42; window 512 8:1 N=5000 106 -> 86.
// The schedule runs on a fixed array, so planning allocates nothing (beyond 1024 key blocks, none of
// which the registry splits, equal splits stay), and a candidate that an even schedule could not
// make shorter is not run. Host time per backward, with a heap-allocated schedule before -> now:
// D=512 2 x 16:2 N=2048 5.4 -> 2.8, 8:1 N=8192 23 -> 6.6, N=16384 84 -> 13, D=64 8:1 N=65536 288 -> 31 us.
struct DkvPlan {
  int chunk;
  int nblocks;
};  // chunk 0: equal splits

constexpr int kPlanBlocks = 1024;    // key blocks
constexpr int kPlanSteps = 1 << 15;  // time steps of one workgroup

inline DkvPlan plan_dkv(const BwdDkvParams& p, int wgs_per_cu) {
  const int slots = 256 * wgs_per_cu;
  const int copies = p.B * p.Hkv;  // grids of key blocks
  if (p.n_kb > kPlanBlocks) return DkvPlan{0, 0};
  int iterations[kPlanBlocks];  // never increasing: a later key block is seen by fewer query tiles
  int64_t work = 0;
  for (int kb = 0; kb < p.n_kb; ++kb) work += iterations[kb] = dkv_iterations(p, kb * p.wkv);
  const int longest = std::max(1, iterations[0]);
  auto longer_than = [&](int64_t x) {  // key blocks of more than x iterations
    return (int)(std::partition_point(iterations, iterations + p.n_kb, [&](int n) { return n > x; }) - iterations);
  };
  auto count = [&](int chunk) {
    if (chunk == 0) return (int64_t)p.n_kb * p.q_splits * copies;
    int64_t c = p.n_kb;
    for (int j = 1; j < p.q_splits; ++j) c += longer_than((int64_t)j * chunk);
    return c * copies;
  };
  auto partials = [&](int chunk) {  // workgroups of key blocks with two splits or more
    return count(chunk) - (chunk == 0 ? 0 : (int64_t)(p.n_kb - longer_than(chunk)) * copies);
  };
  // List schedule: free_at[t % ring] of the slots become free at time t, all of them within one
  // workgroup's length of `now`. A step is an iteration, or 2^unit where a workgroup has more than
  // the array holds.
  uint16_t free_at[kPlanSteps];
  auto cost = [&](int chunk) {
    auto splits = [&](int kb) { return dkv_splits_of(iterations[kb], chunk, p.q_splits); };
    auto length = [&](int kb, int c) { return (iterations[kb] + c - 1) / c + 8; };
    int most = 0;
    for (int kb = 0; kb < p.n_kb; ++kb) most = std::max(most, length(kb, splits(kb)));
    int unit = 0, ring = 1;
    while ((most >> unit) + 1 >= kPlanSteps) ++unit;
    while (ring <= (most >> unit) + 1) ring *= 2;
    std::fill(free_at, free_at + ring, (uint16_t)0);
    free_at[0] = (uint16_t)slots;
    int now = 0, end = 0;
    for (int kb = 0; kb < p.n_kb; ++kb) {
      const int c = splits(kb), len = (length(kb, c) + (1 << unit) - 1) >> unit;
      for (int64_t left = (int64_t)c * copies; left > 0;) {
        while (free_at[now & (ring - 1)] == 0) ++now;
        const int n = (int)std::min<int64_t>(left, free_at[now & (ring - 1)]);
        free_at[now & (ring - 1)] -= (uint16_t)n;
        free_at[(now + len) & (ring - 1)] += (uint16_t)n;
        end = std::max(end, now + len);
        left -= n;
      }
    }
    return (double)((int64_t)end << unit) + 0.03 * (double)partials(chunk);
  };
  double best_cost = cost(0);
  DkvPlan best{0, (int)count(0)};
  const int least = (longest + p.q_splits - 1) / p.q_splits;
  for (int halves = 2; halves <= 4; ++halves) {
    const int64_t most = (int64_t)slots * halves / 2;
    int lo = least, hi = longest;  // the shortest chunk with at most `most` workgroups, or one split each
    while (lo < hi) {
      const int mid = (lo + hi) / 2;
      if (count(mid) <= most) {
        hi = mid;
      } else {
        lo = mid + 1;
      }
    }
    const double even = (double)(work * copies + 8 * count(lo)) / slots + 0.03 * (double)partials(lo);
    if (even >= best_cost) continue;
    const double c = cost(lo);
    if (c < best_cost) {
      best_cost = c;
      best = {lo, (int)count(lo)};
    }
  }
  return best;
}

}  // namespace gfa
