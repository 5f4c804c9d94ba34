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
//   * where trees start as chains (cc.hip hooks every vertex under its smallest
//     neighbour), a find of more than kFindMark hops also stores the ancestor it has
//     reached, into its own start vertex and so without a queue.  The finds that pass there
//     take that far a hop, and the whole chain's finds, all under way at once, end
//     after a number of steps that is its length's logarithm instead of its root: paths
//     of 2^16 and 2^20 vertices and a ring of 2^22 0.284, 1.42 and 5.06 ms without
//     the marks, 0.061, 0.255 and 0.88 with them (path halving: 0.108, 0.73 and 2.5), meshes of
//     65536 x 16 and 16 x 65536 0.249 and 0.356 -> 0.140 and 0.121, road 2048^2 0.82
//     either way (marks from 8 and 32 hops on: 0.91 and 0.86; the path of 2^20 0.27 and
//     0.30).  The edge form and the gangs of a batch start from single vertices and
//     do without (a gang of one on the 16384 x 64 mesh 31 ms, with marks 50).
#pragma once

#include "device_common.hpp"
#include "find_walk.hpp"

namespace indigo {

constexpr int kFindDepth = 5;
constexpr int kFindMark = 64;

// Root of x.
template <int kDepth = kFindDepth, int kMark = 0>
IG_DEV int find_root(int* parent, int x)
{
  return find_walk<kDepth, kMark>(
      x, [parent](int v) { return ld_relaxed(&parent[v]); }, [parent](int v, int p) { st_relaxed(&parent[v], p); });
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
template <int kDepth = kFindDepth, int kMark = 0>
IG_DEV void link(int* parent, int a, int b)
{
  int ra = find_root<kDepth, kMark>(parent, a);
  int rb = find_root<kDepth, kMark>(parent, b);
  while (ra != rb) {
    const int hi = ra > rb ? ra : rb;
    const int lo = ra > rb ? rb : ra;
    const int now = hook(parent, hi, lo);
    if (now == hi) return;
    // climb from where hi now points
    ra = find_root<kDepth, kMark>(parent, ra == hi && now >= 0 ? now : ra);
    rb = find_root<kDepth, kMark>(parent, rb == hi && now >= 0 ? now : rb);
  }
}

}  // namespace indigo
