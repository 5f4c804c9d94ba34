// Breadth-first search (hop distance from one source) on gfx950.
//
// Reference semantics: GPUbfs_vertex / GPUbfs_edge (include/bfs_vertex_cuda.h:61,
// include/bfs_edge_cuda.h:61); dist[v] = number of hops from src, INT_MAX when
// unreachable; the result equals CPUserialDijkstra with unit weights
// (include/bfs_vertex_cuda.h:75-99).
//
// Design: one persistent kernel runs every level; levels are
// separated by the bounded grid barrier (coherent mode: dist, queues and
// counters are only touched with device-scope atomic accesses), so the host
// never round-trips per
// level (the reference copies a goagain flag D2H every level,
// e.g. codes/cuda/bfs-cuda/BFS_CUDA_V_Topo_Push_Determ_IntType_ReadModifyWrite_
// NonPersist_Atomic_Thread_NoBoundsBug2_NoBoundsBug1.cu:98-106).
// Each level is either
//   * top-down: the degree-binned frontier of frontier.hpp (small lists by
//     64-lane waves with the in-wave balancer, mid lists one wave each, huge
//     lists in 512-entry items of one wave each); a neighbour is claimed
//     with one CAS INT_MAX -> L+1, so each vertex joins the next frontier
//     exactly once; or
//   * bottom-up: every unvisited vertex looks for a parent with dist == L and
//     stops at the first one (Beamer, Asanovic, Patterson, SC'12): short
//     lists one lane each in vertex order, long lists (collected once at
//     start) one wave each with a ballot per 64 entries.
// The direction follows Beamer's heuristic (m_f > m_u / 14 -> bottom-up,
// n_f < V / 24 -> top-down), evaluated identically by every workgroup.
// Narrow frontiers (high-diameter graphs) are advanced by one workgroup or a
// team of them, with LDS queues and no grid barriers (team_phase).  Vertices without
// neighbours get their level but never enter a frontier.
#include "bfs.hpp"

#include "by_pass.hpp"
#include "frontier.hpp"
#include "team.hpp"
#include "trace.hpp"

namespace indigo {

namespace {

constexpr int kBfsBlock = 512;
// Team phase: LDS capacity of a member's share, in vertices and in the degree
// sum (an upper bound on its next share).
constexpr int kSmallCap = 2048;
// Degree sums up to which a frontier is one workgroup's, and a member's average
// share of a team's.  (One workgroup for up to 2047 entries made a 300 x 411 road
// 2.11 ms instead of 1.58; shares of 512 measured the same as 1024.)  A team also
// takes only a frontier at most twice as large as the one before: on a graph
// whose levels explode, it would have to hand the next one back at once.
constexpr unsigned kSoloEntries = 1024;
constexpr unsigned kShareEntries = 1024;

// Largest share with which a team goes on: one workgroup hands over to the
// grid (and a team) above kSoloEntries, a team when a member's LDS may not hold
// the next share.
IG_DEV unsigned team_share(int size) { return size == 1 ? kSoloEntries : static_cast<unsigned>(kSmallCap); }

struct BfsBase {
  int level;
  unsigned last_m;
};

struct BfsControl {
  GridBarrier bar;
  TeamSlots team;
  FrontierCounters cnt[3];
  FrontierCounters heavy;  // static lists of >= kMidDeg entries (bottom-up)
  int levels;
  int bottom_up_levels;
  int small_levels;
  int status;
  // where the grid resumes after a team phase: level, degree sum of the level before it
  ByPass<BfsBase> base;
  int pad[24];
  LevelTrace trace;
};

struct BfsArgs {
  int nodes;
  int edges;
  int src;
  int allow_bu;
  int allow_small;
  const int* __restrict__ nindex;
  const int* __restrict__ nlist;
  int* dist;
  FrontierQueues fq[2];
  FrontierQueues heavy;
  BfsControl* ctl;
  long long budget;
  long long start_ticks;
};

IG_DEV int degree_of(const int* __restrict__ nindex, int u) { return nindex[u + 1] - nindex[u]; }

// Claims u for level `next` if unvisited; exactly one caller wins.
IG_DEV bool claim(int* dist, int u, int next)
{
  return dist[u] == kInf && cas_relaxed(&dist[u], kInf, next);
}

IG_DEV void top_down(const BfsArgs& a, int L, const FrontierCounters& ic, const FrontierQueues& in,
                     const FrontierQueues& out, FrontierCounters* oc, FrontierEmitter& E)
{
  const int next = L + 1;
  auto visit = [&](int, int e, bool active) {
    bool won = false;
    int u = 0, udeg = 0;
    if (active) {
      u = a.nlist[e];
      won = claim(a.dist, u, next);
      if (won) udeg = degree_of(a.nindex, u);
    }
    frontier_emit_block(E, won && udeg > 0, u, udeg, out, oc);
  };
  expand_huge(in, huge_count(ic.hpack), huge_chunks(ic.hpack), a.nindex, visit);
  expand_mid(in, ic.nm, a.nindex, visit);
  const unsigned avg = ic.nm == 0 && ic.hpack == 0 ? static_cast<unsigned>(ic.m / ic.n) : 16u;
  expand_small(in.q, ic.n, a.nindex, visit, small_share(ic.n, avg));
}

IG_DEV void bottom_up(const BfsArgs& a, int L, unsigned nheavy, const FrontierQueues& out, FrontierCounters* oc,
                      FrontierEmitter& E)
{
  const int next = L + 1;
  const int lane = lane_id();
  // short lists: one lane per vertex, vertex order
  const int stride = gridDim.x * blockDim.x;
  for (int base = blockIdx.x * blockDim.x; base < a.nodes; base += stride) {
    const int v = base + static_cast<int>(threadIdx.x);
    bool found = false;
    int deg = 0;
    if (v < a.nodes && ld_relaxed(&a.dist[v]) == kInf) {
      const int beg = a.nindex[v], end = a.nindex[v + 1];
      deg = end - beg;
      if (deg < kMidDeg) {
        for (int e = beg; e < end; e++) {
          if (ld_relaxed(&a.dist[a.nlist[e]]) == L) {
            found = true;
            break;
          }
        }
        if (found) st_relaxed(&a.dist[v], next);
      }
    }
    frontier_emit_block(E, found, v, deg, out, oc);
  }
  // long lists: one wave per vertex, 64 entries per ballot
  const int wpb = blockDim.x / kWave;
  for (unsigned i = blockIdx.x * wpb + threadIdx.x / kWave; i < nheavy; i += gridDim.x * wpb) {
    const int v = ld_relaxed(&a.heavy.mq[i]);
    if (ld_relaxed(&a.dist[v]) != kInf) continue;
    const int beg = a.nindex[v], end = a.nindex[v + 1];
    bool found = false;
    for (int base = beg; base < end; base += kWave) {
      const int e = base + lane;
      if (__ballot(e < end && ld_relaxed(&a.dist[a.nlist[e]]) == L) != 0) {
        found = true;
        break;
      }
    }
    if (found && lane == 0) st_relaxed(&a.dist[v], next);
    frontier_emit_block(E, found && lane == 0, v, end - beg, out, oc);
  }
}

// LDS of the team phase (shares the kernel's LDS with the level emitter, which
// is idle meanwhile).
struct SmallLds {
  TeamShare<kSmallCap> share;
  PhaseStop stop;
};

// A team of workgroups (one, or up to kTeamMax) advances levels alone while
// the frontier's lists are short and few: team.hpp has the scheme.  To the grid
// the phase is one pass like any other: entered at level L with the frontier in
// `in` (n vertices of the small queue), it leaves the frontier of the level that
// it reached (empty, or too large for the members) in `out` / `oc`, so the
// workgroups outside the team go straight to the barrier.  A team whose members'
// shares do not all fit the LDS changes nothing and returns L.  Returns the
// level reached; *last gets the degree sum of the level before it.
//
// A level is two dependent rounds of global accesses: the list entries, and
// then, together, each entry's claim (a CAS INT_MAX -> L + 1, so each vertex is
// claimed once) and its neighbour's index pair, which the next level finds in
// LDS.  A slot's list is walked by g lanes, g the power of two that spreads
// the share over the workgroup (64 at most), 4 entries in flight
// per lane; a share averages kSmallCap / slots entries a slot at most, so
// no lane walks long.  (A workgroup prefix sum and a binary search in LDS for each
// entry's owner, on one workgroup, had made a level 10 us on the 1024^2 grid; wider
// frontiers ran on the grid, 8 to 15 us a level.)  1024^2 grid 16.4 -> 6.3 ms a call,
// roads of 1024^2, 2048^2 and 4096^2 28, 40 and 110 -> 5.8, 10.0 and 29.6 ms.
// Claimed vertices join the next frontier whatever their degree; those
// without neighbours contribute no entries and are not handed back.
IG_DEV int team_phase(const BfsArgs& a, int L, unsigned n, const Team& tm, const FrontierQueues& in,
                      const FrontierQueues& out, FrontierCounters* oc, BfsControl* ctl, long long deadline,
                      bool* aborted, unsigned* last, SmallLds& S)
{
  constexpr int kFly = 4;  // entries in flight per lane
  const int t = static_cast<int>(threadIdx.x);
  TeamShare<kSmallCap>& F = S.share;
  if (t == 0) S.stop.clear();
  unsigned entries = 0;
  int cn = share_load(F, L & 1, tm, static_cast<int>(n), a.nindex, [&](int i) { return ld_relaxed(&in.q[i]); }, &entries);
  TeamSum sum;
  *aborted = !team_exchange(&ctl->team, kSlotEntry, tm, static_cast<unsigned>(L) + 1u, entries, 0u, &ctl->bar,
                            deadline, F, sum);
  // (a share of more vertices than the LDS holds has more entries, too: the
  // queue's lists are not empty)
  if (*aborted || sum.most > static_cast<unsigned>(kSmallCap)) return L;
  for (;;) {
    if ((L & 63) == 0 && t == 0) S.stop.post(L, kernel_aborted(&ctl->bar, deadline));
    int shift = 0;  // g = 1 << shift lanes per slot
    while (shift < 6 && (cn << (shift + 1)) <= kBfsBlock) shift++;
    const int sub = t & ((1 << shift) - 1);
    const int now = L & 1, next = L + 1;
    if (t == 0) F.cnt[(L + 2) % 3] = 0ull;
    for (int i0 = 0; i0 < cn; i0 += kBfsBlock >> shift) {
      const int i = i0 + (t >> shift);
      const int beg = i < cn ? F.beg[now][i] : 0;
      const int end = i < cn ? beg + F.deg[now][i] : 0;
      for (int e0 = beg + sub; __ballot(e0 < end) != 0ull; e0 += kFly << shift) {
        int u[kFly];
        IndexPair ip[kFly];
        bool act[kFly];
#pragma unroll
        for (int q = 0; q < kFly; q++) {
          const int e = e0 + (q << shift);
          act[q] = e < end;
          u[q] = act[q] ? a.nlist[e] : 0;
        }
#pragma unroll
        for (int q = 0; q < kFly; q++) {
          if (act[q]) ip[q] = index_pair(a.nindex, u[q]);
          act[q] = act[q] && cas_relaxed(&a.dist[u[q]], kInf, next);
        }
        // (at most as many claims as the share has entries)
        share_append(F, next, act, u, ip);
      }
    }
    __syncthreads();
    if (S.stop.at(L)) {
      *aborted = true;
      return L;
    }
    L = next;
    *last = sum.total;
    const unsigned long long c = F.cnt[L % 3];
    cn = static_cast<int>(c & 0xffffffffull);
    if (!team_exchange(&ctl->team, kSlotLevel + (L & 1), tm, static_cast<unsigned>(L), static_cast<unsigned>(c >> 32),
                       static_cast<unsigned>(cn), &ctl->bar, deadline, F, sum) ||
        (share_uneven(tm, sum) &&
         !share_deal(&ctl->team, L & 1, tm, static_cast<unsigned>(L), out.mq, a.nindex, &ctl->bar, deadline, F, cn, sum))) {
      *aborted = true;
      return L;
    }
    if (sum.total == 0u || sum.most > team_share(tm.size)) break;
  }
  for (int base = 0; base < cn; base += blockDim.x) {
    const int i = base + t;
    const int d = i < cn ? F.deg[L & 1][i] : 0;
    frontier_emit(d > 0, i < cn ? F.v[L & 1][i] : 0, d, out, oc);
  }
  return L;
}

__global__ __launch_bounds__(kBfsBlock) __attribute__((amdgpu_waves_per_eu(6, 8))) void bfs_kernel(BfsArgs a)
{
  // the set-up's heavy-list collection needs a larger mid buffer than the
  // level emitter (no spills to the global counter); they share the LDS
  __shared__ union {
    FrontierEmitter emit;
    HeavyCollector collect;
    SmallLds small;
  } s_lds;
  FrontierEmitter& s_emit = s_lds.emit;
  BfsControl* ctl = a.ctl;
  if (!residency_barrier(&ctl->bar, a.start_ticks)) return;
  const long long deadline = now_ticks() + a.budget;
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  const int stride = gridDim.x * blockDim.x;
  if (tid == 0) ctl->trace.start = now_ticks();
  for (int i = tid; i < a.nodes; i += stride) st_relaxed(&a.dist[i], (i == a.src) ? 0 : kInf);
  if (a.allow_bu) collect_heavy<kMidDeg, INT_MAX, kHugeChunk>(s_lds.collect, a.nodes, a.nindex, a.heavy, &ctl->heavy);
  if (blockIdx.x == 0 && threadIdx.x < kWave) {
    const int deg = degree_of(a.nindex, a.src);
    frontier_emit(threadIdx.x == 0 && deg > 0, a.src, deg, a.fq[0], &ctl->cnt[0]);
  }
  if (!grid_barrier<true>(&ctl->bar, deadline)) {
    if (tid == 0) ctl->status = 1;
    return;
  }
  const unsigned nheavy = ld_relaxed(&ctl->heavy.nm);
  bool bu = false;
  unsigned long long seen_edges = 0;
  int bu_levels = 0;
  int L = 0;
  int R = 0;              // pass: counters rotate and queues alternate by it
  int declined = -1;      // level that a team has left to the grid
  unsigned long long prev = 0;  // degree sum of the level before L
  for (;;) {
    const FrontierCounters ic = counters_load(&ctl->cnt[R % 3]);
    const unsigned long long nf = static_cast<unsigned long long>(ic.n) + ic.nm + huge_count(ic.hpack);
    if (nf == 0) break;
    if (declined != L) seen_edges += ic.m;
    if (a.allow_bu) {
      const unsigned long long e = static_cast<unsigned long long>(a.edges);
      const unsigned long long mu = e > seen_edges ? e - seen_edges : 0ull;
      if (!bu) {
        if (ic.m * 14ull > mu) bu = true;
      } else if (nf * 24ull < static_cast<unsigned long long>(a.nodes)) {
        bu = false;
      }
    }
    int team = 0;  // workgroups of a team phase, 0: a grid level
    if (!bu && a.allow_small && declined != L && ic.nm == 0 && ic.hpack == 0) {
      const int limit = team_limit();
      if (ic.m <= kSoloEntries) team = 1;
      else if (limit > 1 && ic.m <= static_cast<unsigned long long>(limit) * kShareEntries && ic.m <= 2ull * prev)
        team = limit;
    }
    prev = ic.m;
    trace_level(&ctl->trace, L, static_cast<unsigned>(nf), ic.m, team != 0 ? 2 : (bu ? 1 : 0));
    if (tid == 0) counters_clear(&ctl->cnt[(R + 2) % 3]);
    const FrontierQueues& in = a.fq[R & 1];
    const FrontierQueues& out = a.fq[(R + 1) & 1];
    FrontierCounters* oc = &ctl->cnt[(R + 1) % 3];
    if (team != 0) {
      // the workgroups outside the team wait at the next barrier
      const Team tm = make_team(team);
      if (tm.rank >= 0) {
        bool aborted = false;
        unsigned last = 0;
        const int L2 = team_phase(a, L, ic.n, tm, in, out, oc, ctl, deadline, &aborted, &last, s_lds.small);
        if (aborted) {  // (the same in all of a workgroup)
          if (tid == 0) ctl->status = 1;
          return;
        }
        if (tm.rank == 0 && threadIdx.x == 0) {
          st_relaxed(&ctl->base.of(R).level, L2);
          st_relaxed(&ctl->base.of(R).last_m, last);
          ctl->small_levels += L2 - L;
        }
      }
      if (!grid_barrier<true>(&ctl->bar, deadline)) {
        if (tid == 0) ctl->status = 1;
        return;
      }
      const int L2 = ld_relaxed(&ctl->base.of(R).level);
      if (L2 == L) {  // an uneven frontier: this level goes to the grid
        declined = L;
        continue;
      }
      prev = ld_relaxed(&ctl->base.of(R).last_m);
      L = L2;
      R++;
      continue;
    }
    fe_reset(s_emit);
    if (bu) {
      bottom_up(a, L, nheavy, out, oc, s_emit);
      bu_levels++;
    } else {
      top_down(a, L, ic, in, out, oc, s_emit);
    }
    fe_flush(s_emit, out, oc);
    if (!grid_barrier<true>(&ctl->bar, deadline)) {
      if (tid == 0) ctl->status = 1;
      return;
    }
    L++;
    R++;
  }
  if (tid == 0) {
    ctl->levels = L;
    ctl->bottom_up_levels = bu_levels;
  }
}

}  // namespace

// Workgroups of one call, per square root of the entries: R-MAT 12, 14, 16 and 18
// took 0.096, 0.107, 0.117 and 0.173 ms on the whole grid, 0.092, 0.105, 0.114 and
// 0.165 to 0.172 on 64, 128, 256 and 256 to 512 workgroups.
constexpr double kBfsGridPerRoot = 0.2;

size_t bfs_workspace_bytes(int nodes)
{
  const size_t v = static_cast<size_t>(nodes);
  return Carver::round(sizeof(BfsControl)) + 12 * Carver::round(v * 4) + 4096;
}

int bfs_run(indigo_ctx* ctx, int nodes, int edges, const int* nindex, const int* nlist, int src, int* dist,
            BfsStats* stats)
{
  IG_TRY(ensure_workspace(ctx, bfs_workspace_bytes(nodes)));
  IG_TRY(ensure_host_pinned(ctx, sizeof(BfsControl)));
  Carver cv(ctx->ws);
  BfsArgs a{};
  a.ctl = cv.take<BfsControl>(1);
  for (int k = 0; k < 3; k++) {
    FrontierQueues& f = k < 2 ? a.fq[k] : a.heavy;
    f.q = cv.take<int>(nodes);
    f.mq = cv.take<int>(nodes);
    f.hq = cv.take<int>(nodes);
    f.hoff = cv.take<unsigned>(nodes);
  }
  a.nodes = nodes;
  a.edges = edges;
  a.src = src;
  a.allow_bu = ctx->hints[INDIGO_HINT_BFS_DIRECTION] != 1;
  a.allow_small = ctx->hints[INDIGO_HINT_SMALL_FRONTIER] != 1;
  a.nindex = nindex;
  a.nlist = nlist;
  a.dist = dist;
  a.budget = budget_ticks(ctx);
  a.start_ticks = residency_ticks(ctx);
  IG_TRY(zero_async(ctx, a.ctl, sizeof(BfsControl)));
  void* args[] = {&a};
  int grid = 0;
  IG_TRY(coop_launch(ctx, reinterpret_cast<const void*>(bfs_kernel), kBfsBlock, 0, args,
                     graph_grid(nodes, edges, kBfsGridPerRoot), &grid, "bfs_kernel"));
  if (stats) {
    stats->launches = 2;
    stats->grid = grid;
  }
  return INDIGO_OK;
}

int bfs_collect(indigo_ctx* ctx, BfsStats* stats)
{
  Carver cv(ctx->ws);
  BfsControl* ctl = cv.take<BfsControl>(1);
  BfsControl* h = static_cast<BfsControl*>(ctx->host_pinned);
  IG_HIP_TRY(hipMemcpyAsync(h, ctl, sizeof(BfsControl), hipMemcpyDeviceToHost, ctx->stream));
  IG_HIP_TRY(hipStreamSynchronize(ctx->stream));
  IG_TRY(check_abort(ctx, reinterpret_cast<const void*>(bfs_kernel), h->bar.abort.v, "bfs"));
  if (h->status != 0)
    return set_error(INDIGO_ERR_TIMEOUT, "bfs: persistent kernel stopped (status %d) before finishing", h->status);
  if (stats) {
    stats->levels = h->levels;
    stats->bottom_up_levels = h->bottom_up_levels;
    stats->small_levels = h->small_levels;
  }
  store_trace(ctx, h->trace);
  return INDIGO_OK;
}

}  // namespace indigo
