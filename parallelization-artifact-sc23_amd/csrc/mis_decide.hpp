// MIS: one vertex's decision, by a lane or a group of lanes, shared by the
// single-query kernel and the batched engine.  The arguments `a` hold nlist, status
// and flip (see mis.hip).
#pragma once

#include "device_common.hpp"

namespace indigo {

constexpr int kUndecided = 0, kIncluded = 1, kExcluded = 2;
constexpr int kMisLaneUnroll = 4;  // entries per lane and step of a decision
constexpr int kMisGroupShift = 3;  // log2 of the lanes that finish a list a lane has started

IG_DEV unsigned long long mis_key(int v, unsigned flip)
{
  const unsigned p = mis_hash(static_cast<unsigned>(v) + 712313887u) ^ flip;
  return (static_cast<unsigned long long>(p) << 32) | static_cast<unsigned>(v);
}

// One lane decides vertex v from the first kMisLaneUnroll entries of its (short)
// list.  Returns the new state, or -1 if it takes the rest of the list.
template <typename A>
IG_DEV int decide_lane(const A& a, int v, int beg, int end)
{
  // Only neighbours with a larger key can decide v: a smaller one cannot be
  // included while v is undecided (it would need v excluded first), so their
  // states are not read.  The entries' loads are in flight together and
  // evaluated in entry order.
  const unsigned long long kv = mis_key(v, a.flip);
  int u[kMisLaneUnroll], su[kMisLaneUnroll];
#pragma unroll
  for (int q = 0; q < kMisLaneUnroll; q++) u[q] = beg + q < end ? a.nlist[beg + q] : v;
#pragma unroll
  for (int q = 0; q < kMisLaneUnroll; q++)
    su[q] = u[q] != v && mis_key(u[q], a.flip) > kv ? ld_relaxed(&a.status[u[q]]) : kExcluded;
#pragma unroll
  for (int q = 0; q < kMisLaneUnroll; q++) {
    if (su[q] == kIncluded) return kExcluded;
    if (su[q] == kUndecided) return kUndecided;
  }
  return end - beg > kMisLaneUnroll ? -1 : kIncluded;
}
// v, whose list ends within the first step, has just been included: its larger-key
// neighbours are all excluded already, so only the smaller-key ones are read, and
// the undecided among them excluded.  (Storing unconditionally is slower:
// device-scope stores to already excluded hub neighbours cost more than the reads
// they save.)
template <typename A>
IG_DEV void exclude_neighbours_lane(const A& a, int v, int beg, int end)
{
  const unsigned long long kv = mis_key(v, a.flip);
  int u[kMisLaneUnroll], su[kMisLaneUnroll];
#pragma unroll
  for (int q = 0; q < kMisLaneUnroll; q++) u[q] = beg + q < end ? a.nlist[beg + q] : v;
#pragma unroll
  for (int q = 0; q < kMisLaneUnroll; q++)
    su[q] = u[q] != v && mis_key(u[q], a.flip) < kv ? ld_relaxed(&a.status[u[q]]) : kExcluded;
#pragma unroll
  for (int q = 0; q < kMisLaneUnroll; q++)
    if (su[q] == kUndecided) st_relaxed(&a.status[u[q]], kExcluded);
}

// The two together for a vertex per group of 1 << gs lanes (same v, beg, end in a
// group; beg = end where there is none; the entries before from have decided nothing), four entries per lane in flight; all
// lanes of the wave must be converged.  Returns the new state.
template <typename A>
IG_DEV int decide_group(const A& a, int v, int beg, int from, int end, int gs)
{
  const unsigned long long kv = mis_key(v, a.flip);
  const int lane = lane_id();
  const int sub = lane & ((1 << gs) - 1);
  const unsigned long long group = (gs == 6 ? ~0ull : (1ull << (1 << gs)) - 1ull) << (lane - sub);
  int r = beg < end ? -1 : kIncluded;
  for (int e0 = from + sub; __ballot(r < 0) != 0ull; e0 += kMisLaneUnroll << gs) {
    int su[kMisLaneUnroll];
#pragma unroll
    for (int q = 0; q < kMisLaneUnroll; q++) {
      const int e = e0 + (q << gs);
      const int u = r < 0 && e < end ? a.nlist[e] : v;
      su[q] = u != v && mis_key(u, a.flip) > kv ? ld_relaxed(&a.status[u]) : kExcluded;
    }
    bool inc = false, hi = false;
#pragma unroll
    for (int q = 0; q < kMisLaneUnroll; q++) {
      inc |= su[q] == kIncluded;
      hi |= su[q] == kUndecided;
    }
    const unsigned long long incs = __ballot(inc) & group, his = __ballot(hi) & group;
    if (r < 0) {
      if (incs != 0ull) r = kExcluded;
      else if (his != 0ull) r = kUndecided;
      else if (e0 - sub + (kMisLaneUnroll << gs) >= end) r = kIncluded;
    }
  }
  if (beg < end && r != kUndecided && sub == 0) st_relaxed(&a.status[v], r);
  if (r == kIncluded) {
    for (int e0 = beg + sub; e0 < end; e0 += kMisLaneUnroll << gs) {
      int u[kMisLaneUnroll], su[kMisLaneUnroll];
#pragma unroll
      for (int q = 0; q < kMisLaneUnroll; q++) u[q] = e0 + (q << gs) < end ? a.nlist[e0 + (q << gs)] : v;
#pragma unroll
      for (int q = 0; q < kMisLaneUnroll; q++)
        su[q] = u[q] != v && mis_key(u[q], a.flip) < kv ? ld_relaxed(&a.status[u[q]]) : kExcluded;
#pragma unroll
      for (int q = 0; q < kMisLaneUnroll; q++)
        if (su[q] == kUndecided) st_relaxed(&a.status[u[q]], kExcluded);
    }
  }
  return r;
}

}  // namespace indigo
