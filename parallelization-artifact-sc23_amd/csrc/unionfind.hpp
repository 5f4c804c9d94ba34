// Concurrent union-find on a parent array, shared by the CC kernels.
//
// Every link hooks the LARGER root under the smaller one with a CAS, so
// parent[x] <= x always holds and each final root is the minimum id of its
// tree - once all edges are linked, the minimum id of its component, which
// is the reference's CC label (min-label propagation to a fixed point,
// e.g. codes/cuda/cc-cuda/CC_CUDA_V_Topo_Push_NonDeterm_IntType_
// ReadModifyWrite_NonPersist_Atomic_Thread_NoBoundsBug2_NoBoundsBug1.cu:47-76).
//
// What bounds it is writes to one address, which follow one another at about
// 10 ns each: random graphs (2^20 vertices, degree 16) took 2.6 to 4.4 ms a call,
// roads of 2048^2 2.4, with nearly all of it in such queues.  So
//   * a find stores nothing on the way, only the root into the vertex it started
//     from, and only from depth kFindDepth on (halving the path made every find
//     write the few vertices below the root);
//   * a root is read again before its CAS, and of a wave's lanes that hook the
//     same root only the first tries (when large trees meet, lanes all over
//     the grid find the same two roots at once).
// 0.39 to 0.44 and 0.87 ms; 4-neighbour grid of 1024^2 0.67 -> 0.22.  Depths of 1,
// 2 and 5 gave 0.83, 0.64 and 0.42 ms on the random graph, 0.225, 0.245 and 0.250
// on R-MAT 22 (the gangs of a batch, whose vertices fewer lanes share, take 2).
#pragma once

#include "device_common.hpp"

namespace indigo {

constexpr int kFindDepth = 5;

// Root of x.  The store replaces x's parent by one of its ancestors, so
// concurrent finds and links stay valid (x is no root, so no link writes it).
template <int kDepth = kFindDepth>
IG_DEV int find_root(int* parent, int x)
{
  int r = x, p = ld_relaxed(&parent[x]);
  int hops = 0;
  while (p != r) {
    r = p;
    p = ld_relaxed(&parent[r]);
    hops++;
  }
  if (hops > kDepth) st_relaxed(&parent[x], r);
  return r;
}

// Hooks root hi under lo.  Returns hi on success, where hi points by now if it is
// no root any more, and -1 if this lane left the try to another.
IG_DEV int hook(int* parent, int hi, int lo)
{
  const bool shared = hi == __builtin_amdgcn_readfirstlane(hi);
  const bool first = lane_id() == __builtin_amdgcn_readfirstlane(lane_id());
  int seen = ld_relaxed(&parent[hi]);
  if (seen != hi) return seen;
  if (shared && !first) return -1;
  __hip_atomic_compare_exchange_strong(&parent[hi], &seen, lo, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  return seen;
}

// Joins the trees of a and b.  (Each round the first lane of every wave that still
// has something to join either joins it or finds that another wave has.)
template <int kDepth = kFindDepth>
IG_DEV void link(int* parent, int a, int b)
{
  int ra = find_root<kDepth>(parent, a);
  int rb = find_root<kDepth>(parent, b);
  while (ra != rb) {
    const int hi = ra > rb ? ra : rb;
    const int lo = ra > rb ? rb : ra;
    const int now = hook(parent, hi, lo);
    if (now == hi) return;
    // climb from where hi now points
    ra = find_root<kDepth>(parent, ra == hi && now >= 0 ? now : ra);
    rb = find_root<kDepth>(parent, rb == hi && now >= 0 ? now : rb);
  }
}

}  // namespace indigo
