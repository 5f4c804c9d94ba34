// A team of workgroups that advances narrow levels of a traversal by itself
// while the rest of a persistent grid waits at its barrier.
//
// Each member keeps its share of the frontier in its own LDS and expands it
// itself: what a member claims, it expands in the next level.  A level then ends
// with one exchange: every member publishes the size of its next share under the
// level's tag and reads the others' (one wave, one lane per member), which is the
// level's barrier and its frontier total in one.  A store and a poll stand where
// the grid pays its barrier, the queue appends (a global atomic and a store
// round) and the queue reads.  Shares drift apart (on a 2048^2 road one of 32
// grew to 1929 of 6860 entries within 800 levels, and the level's time with it,
// 3.4 to 11.5 us), so the members deal the frontier out again when the largest
// share passes half as much again as the average and 64 entries (share_uneven).
// A team of one is a workgroup alone: its exchange is free.
#pragma once

#include "device_common.hpp"
#include "phase_stop.hpp"

namespace indigo {

constexpr int kTeamMax = 32;  // members at most (one lane each in an exchange)

// Slots of the exchanges, (tag << 32) | value per member.  A level's slots are
// double-buffered by its parity: a member reuses a slot two levels on, when
// every member has passed the exchange in between.  The other buffers serve one
// kind of exchange each.  Tags of one buffer only grow, from phase to phase too.
enum TeamSlot { kSlotLevel = 0, kSlotEntry = 2, kSlotDeal = 3, kSlotDealt = 4, kSlotMin = 5, kSlotKinds = 6 };
struct alignas(128) TeamSlots {
  unsigned long long v[kSlotKinds][kTeamMax];
};

// The calling workgroup's rank in a team (-1: not a member).  Workgroups b with
// b % 8 == 0 are dispatched to one XCD, whose L2 then holds the lists that
// neighbouring members read.
struct Team {
  int size, rank;
};

IG_DEV Team make_team(int size)
{
  const int b = static_cast<int>(blockIdx.x);
  return Team{size, size == 1 ? (b == 0 ? 0 : -1) : ((b & 7) == 0 && (b >> 3) < size ? b >> 3 : -1)};
}

IG_DEV int team_limit()
{
  const int per = static_cast<int>(gridDim.x) >> 3;
  return per < 1 ? 1 : (per < kTeamMax ? per : kTeamMax);
}

// Rank 0's thread 0: waits until every workgroup outside the team has arrived at the
// barrier that ends the pass (the members' all have b % 8 == 0).  Waits no longer once the
// kernel must stop, which the phase's own look finds within 64 turns.
IG_DEV void wait_others(GridBarrier* gb, const Team& tm, long long deadline)
{
  wait_arrived(gb, ((gridDim.x + 7u) >> 3) - static_cast<unsigned>(tm.size), deadline);
}

// What an exchange tells: over all members the entries (sum, maximum) and the
// vertices, and the vertices of lower ranks.
struct TeamSum {
  unsigned total, most, vertices, before;
};

// nindex[u] and nindex[u + 1] in one load (4-byte aligned).
struct __attribute__((packed, aligned(4))) IndexPair {
  int beg, end;
};
IG_DEV IndexPair index_pair(const int* __restrict__ nindex, int u)
{
  return *reinterpret_cast<const IndexPair*>(nindex + u);
}

// A member's share by level parity: vertices with their list bounds.  Sizes
// rotate over three counters, (sum of min(degree, kCap + 1) << 32) | vertices: in
// level L, cnt[(L + 1) % 3] is filled and cnt[(L + 2) % 3] cleared, so a level
// needs one workgroup barrier.  At most kCap vertices and entries.
template <int kCap>
struct TeamShare {
  int v[2][kCap];
  int beg[2][kCap];
  int deg[2][kCap];
  unsigned long long cnt[3];
  TeamSum sum;
  int ok;
};

// One wave's part of an exchange: publishes `value` under `tag`, waits until every
// member has, and returns lane i's member i's value (0 beyond the team).  False in
// *ok when the kernel must stop.
IG_DEV unsigned team_values(TeamSlots* ts, int slot, const Team& tm, unsigned tag, unsigned value, GridBarrier* gb,
                            long long deadline, int* ok)
{
  const int lane = lane_id();
  unsigned long long* slots = ts->v[slot];
  unsigned long long x = static_cast<unsigned long long>(tag) << 32;
  if (lane == 0) st_relaxed(&slots[tm.rank], x | value);
  *ok = 1;
  for (int spin = 1;; spin++) {
    if (lane < tm.size) x = ld_relaxed(&slots[lane]);
    if (__ballot((x >> 32) != tag) == 0ull) break;
    if ((spin & 63) == 0) {
      int stop = 0;
      if (lane == 0) stop = kernel_aborted(gb, deadline) ? 1 : 0;
      if (wave_bcast(stop, 0) != 0) {
        *ok = 0;
        break;
      }
    }
  }
  return static_cast<unsigned>(x & 0xffffffffull);
}

// Workgroup-collective: a barrier of the team that publishes a share's
// `entries` and `vertices` (both uniform, at most 65535).  False when the kernel
// must stop.
template <int kCap>
IG_DEV bool team_exchange(TeamSlots* ts, int slot, const Team& tm, unsigned tag, unsigned entries, unsigned vertices,
                          GridBarrier* gb, long long deadline, TeamShare<kCap>& S, TeamSum& out)
{
  if (tm.size == 1) {
    out = TeamSum{entries, entries, vertices, 0u};
    return true;
  }
  wave_drain();
  __syncthreads();
  if (threadIdx.x < kWave) {
    const int lane = lane_id();
    int ok = 1;
    const unsigned x =
        team_values(ts, slot, tm, tag, (min(entries, 0xffffu) << 16) | vertices, gb, deadline, &ok);
    const unsigned e = x >> 16, n = x & 0xffffu;
    const int incl = wave_inclusive_scan(static_cast<int>(n));
    const unsigned total = wave_sum(e), most = wave_max(e);
    if (lane == tm.rank) S.sum.before = static_cast<unsigned>(incl) - n;
    if (lane == kWave - 1) S.sum.vertices = static_cast<unsigned>(incl);
    if (lane == 0) {
      S.sum.total = total;
      S.sum.most = most;
      S.ok = ok;
    }
  }
  __syncthreads();
  out = S.sum;
  return S.ok != 0;
}

// Workgroup-collective: the members' smallest value (at most INT_MAX).
template <int kCap>
IG_DEV bool team_min(TeamSlots* ts, const Team& tm, unsigned tag, unsigned value, GridBarrier* gb, long long deadline,
                     TeamShare<kCap>& S, unsigned* out)
{
  *out = value;
  if (tm.size == 1) return true;
  wave_drain();
  __syncthreads();
  if (threadIdx.x < kWave) {
    int ok = 1;
    const unsigned x = team_values(ts, kSlotMin, tm, tag, value, gb, deadline, &ok);
    const unsigned least = wave_min(lane_id() < tm.size ? x : 0xffffffffu);
    if (lane_id() == 0) {
      S.sum.total = least;
      S.ok = ok;
    }
  }
  __syncthreads();
  *out = S.sum.total;
  return S.ok != 0;
}

// Workgroup-collective: every size-th vertex of a queue of n into the share of
// parity p (as many as fit), with at(i) its i-th vertex.  Returns the share's
// vertices and entries, fitting or not.
template <int kCap, typename F>
IG_DEV int share_load(TeamShare<kCap>& S, int p, const Team& tm, int n, const int* __restrict__ nindex, F&& at,
                      unsigned* entries)
{
  if (threadIdx.x == 0) {
    S.cnt[0] = 0ull;
    S.cnt[1] = 0ull;
    S.cnt[2] = 0ull;
    S.sum.total = 0u;
  }
  const int cn = (n - tm.rank + tm.size - 1) / tm.size;
  unsigned have = 0;
  for (int i = threadIdx.x; i < cn; i += blockDim.x) {
    const int v = at(i * tm.size + tm.rank);
    const IndexPair ip = index_pair(nindex, v);
    if (i < kCap) {
      S.v[p][i] = v;
      S.beg[p][i] = ip.beg;
      S.deg[p][i] = ip.end - ip.beg;
    }
    have += static_cast<unsigned>(min(ip.end - ip.beg, 0xffff));
    have = min(have, 0xffffu);
  }
  __syncthreads();
  if (have != 0u) atomicAdd(&S.sum.total, have);
  __syncthreads();
  *entries = min(S.sum.total, 0xffffu);
  return cn;
}

// Wave-collective: appends each lane's vertices u[q] with `join` to the share
// of level `next`.  True in a lane that had one left over (the share is full).
template <int kFly, int kCap>
IG_DEV bool share_append(TeamShare<kCap>& S, int next, const bool (&join)[kFly], const int (&u)[kFly],
                         const IndexPair (&ip)[kFly])
{
  unsigned mine = 0;  // (sum of clamped degrees << 10) | vertices
#pragma unroll
  for (int q = 0; q < kFly; q++)
    if (join[q]) mine += (static_cast<unsigned>(min(ip[q].end - ip[q].beg, kCap + 1)) << 10) + 1u;
  static_assert(kFly * kWave < 1024 && (kFly * kWave * (kCap + 1ll)) < (1ll << 22), "fields of `mine`");
  const unsigned incl = static_cast<unsigned>(wave_inclusive_scan(static_cast<int>(mine)));
  const unsigned all = static_cast<unsigned>(wave_bcast(static_cast<int>(incl), kWave - 1));
  if (all == 0u) return false;
  int slot = 0;
  if (lane_id() == 0)
    slot = static_cast<int>(atomicAdd(&S.cnt[next % 3],
                                      (static_cast<unsigned long long>(all >> 10) << 32) | (all & 1023u)));
  slot = wave_bcast(slot, 0) + static_cast<int>((incl & 1023u) - (mine & 1023u));
  const int p = next & 1;
#pragma unroll
  for (int q = 0; q < kFly; q++) {
    if (join[q] && slot < kCap) {
      S.v[p][slot] = u[q];
      S.beg[p][slot] = ip[q].beg;
      S.deg[p][slot] = ip[q].end - ip[q].beg;
    }
    if (join[q]) slot++;
  }
  return mine != 0u && slot > kCap;
}

// Whether the members should deal the frontier out again.
IG_DEV bool share_uneven(const Team& tm, const TeamSum& s)
{
  return tm.size > 1 && s.most > s.total / static_cast<unsigned>(tm.size) * 3u / 2u + 64u;
}

// Workgroup-collective: deals the team's frontier (the shares of parity p) out
// evenly, through `buf` (at least s.vertices ints, idle meanwhile).  cn and s are
// replaced by those of the new shares.
template <int kCap>
IG_DEV bool share_deal(TeamSlots* ts, int p, const Team& tm, unsigned tag, int* buf, const int* __restrict__ nindex,
                       GridBarrier* gb, long long deadline, TeamShare<kCap>& S, int& cn, TeamSum& s)
{
  for (int i = threadIdx.x; i < cn; i += blockDim.x) st_relaxed(&buf[s.before + i], S.v[p][i]);
  const int n = static_cast<int>(s.vertices);
  if (!team_exchange(ts, kSlotDeal, tm, tag, 0u, 0u, gb, deadline, S, s)) return false;
  unsigned entries = 0;
  cn = share_load(S, p, tm, n, nindex, [&](int i) { return ld_relaxed(&buf[i]); }, &entries);
  return team_exchange(ts, kSlotDealt, tm, tag, entries, static_cast<unsigned>(cn), gb, deadline, S, s);
}

}  // namespace indigo
