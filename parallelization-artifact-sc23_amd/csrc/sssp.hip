// Single-source shortest paths (int32 weights and distances) on gfx950.
//
// Reference semantics: GPUsssp_vertex / GPUsssp_edge (include/sssp_vertex_cuda.h:60,
// include/sssp_edge_cuda.h:60): dist[src] = 0, INT_MAX when unreachable,
// relaxations d = dist[v] + w in int arithmetic; results equal the serial
// Dijkstra of sssp_vertex_cuda.h:74-99.
//
// Design: one persistent kernel (coherent-mode barriers: dist,
// stamps, queues, piles and counters only see device-scope atomic accesses)
// running near-far
// label-correcting SSSP (Davidson et al., IPDPS'14):
//   * the near frontier holds vertices whose distance improved below the
//     split T; it is expanded with the degree-binned machinery of
//     frontier.hpp (64-lane in-wave edge balancing, huge lists split over
//     workgroups); each edge relaxes with atomicMin and, on improvement, the
//     target joins the next near frontier (deduplicated per iteration with an
//     exchange on stamp[u]) or, if its distance is >= T, the far pile
//     (deduplicated per epoch with farstamp[u]) while far_min tracks the
//     smallest parked distance;
//   * far piles rotate over three buffers: epoch e files into pile e % 3 and
//     re-files into pile (e + 1) % 3 while pile (e + 2) % 3, consumed one
//     barrier earlier, is cleared - no buffer ever has two roles at once;
//   * when the near frontier empties, the split moves to
//     max(T, far_min) + delta and one pass re-files the far pile: entries
//     below the new split join the near frontier, settled entries (distance
//     below the old split, already expanded at that distance) are dropped,
//     the rest stay parked;
//   * vertices are expanded with their current distance (re-read at
//     expansion), so stale duplicates only cost work, never correctness;
//   * while the near frontier is narrow (only short lists, few entries), one
//     workgroup or a team of them runs the near iterations and the splits
//     alone, with the frontier and the newly parked vertices in LDS and no grid
//     barriers (team_near); it hands both back to the grid when they outgrow
//     the LDS.  Deep sparse graphs spend thousands of iterations on frontiers
//     of tens to thousands of vertices.
// delta defaults to a sampled mean weight x 32 / mean degree (at least 1).
#include "sssp.hpp"

#include "by_pass.hpp"
#include "far_piles.hpp"
#include "frontier.hpp"
#include "team.hpp"
#include "trace.hpp"

namespace indigo {

namespace {

constexpr int kSsspBlock = 512;
// Team phase: LDS capacity of a member's near share, in vertices and in entries,
// and of its far pile; degree sums up to which a near frontier is one
// workgroup's, and a member's average share of a team's.
constexpr int kShareCap = 1024;
constexpr int kFarCap = 2048;
constexpr unsigned kSoloEntries = 1024;
constexpr unsigned kShareEntries = 512;

struct SsspBase {
  int it, split, epoch;
  unsigned last_m;
};

struct SsspControl {
  GridBarrier bar;
  TeamSlots team;
  FrontierCounters cnt[3];
  PaddedU32 far_cnt[3];
  PaddedU32 far_min[3];
  int iterations;
  int epochs;
  int status;
  int delta;
  int small_iters;  // iterations (near and split) run by teams
  // where the grid resumes after a team phase: iteration (stamp) count, split
  // T, far-pile epoch, degree sum of the frontier before the one handed over
  ByPass<SsspBase> base;
  int pad[19];
  LevelTrace trace;
};

struct SsspArgs {
  int nodes;
  int edges;
  int src;
  int delta_hint;
  int allow_small;  // the team phase may run (INDIGO_HINT_SMALL_FRONTIER != 1)
  const int* __restrict__ nindex;
  const int* __restrict__ nlist;
  const int* __restrict__ eweight;
  int* dist;
  int* stamp;
  int* farstamp;
  int* far[3];
  FrontierQueues fq[2];
  SsspControl* ctl;
  long long budget;
  long long start_ticks;
};

IG_DEV int degree_of(const int* __restrict__ nindex, int u) { return nindex[u + 1] - nindex[u]; }

// Relaxes one CSR entry e of v (distance dv) when `active`: an improvement
// below the split T joins the next near frontier (deduplicated per iteration
// by stamp), one at or above T is parked in the far pile (deduplicated per
// epoch by farstamp).  Wave-collective: all lanes converged.
// Workgroup-aggregated emission state of one SSSP phase.
struct SsspEmit {
  FrontierEmitter near;
  BlockQueue<2048> far;
  unsigned far_min;
};

IG_DEV void se_reset(SsspEmit& S)
{
  if (threadIdx.x == 0) S.far_min = static_cast<unsigned>(kInf);
  fe_reset(S.near);
  bq_reset(S.far);
}

IG_DEV void se_park(SsspEmit& S, bool park, int u, int d, int* far, unsigned* far_cnt)
{
  if (__ballot(park) == 0ull) return;
  bq_append(S.far, park, u, far, far_cnt);
  const int m = wave_min(park ? d : kInf);
  if (lane_id() == 0 && m != kInf) atomicMin(&S.far_min, static_cast<unsigned>(m));
}

IG_DEV void se_flush(SsspEmit& S, const FrontierQueues& out, FrontierCounters* oc, int* far, unsigned* far_cnt,
                     unsigned* far_min)
{
  fe_flush(S.near, out, oc);
  bq_flush(S.far, far, far_cnt);
  if (threadIdx.x == 0 && S.far_min != static_cast<unsigned>(kInf)) atomic_min_relaxed(far_min, S.far_min);
  __syncthreads();
}

IG_DEV void relax(const SsspArgs& a, int dv, int e, bool active, int T, int it_stamp, int epoch, int* far,
                  unsigned* far_cnt, SsspEmit& S, const FrontierQueues& out, FrontierCounters* oc)
{
  bool near = false, park = false;
  int u = 0, nd = 0, udeg = 0;
  if (active) {
    u = a.nlist[e];
    nd = dv + a.eweight[e];
    // device-scope read: a plain load may see a stale L2 copy of a distance
    // another XCD has lowered, and let a useless atomic through
    if (nd < ld_relaxed(&a.dist[u])) {
      // the minimum, the dedup exchange and the degree leave together: a
      // lane whose check passed may join u whether or not its own atomicMin
      // was the one that lowered dist[u] - someone did, in this iteration
      const bool below = nd < T;
      atomic_min_relaxed(&a.dist[u], nd);
      int* mark = below ? &a.stamp[u] : &a.farstamp[u];
      const int tag = below ? it_stamp : epoch;
      const int seen = __hip_atomic_exchange(mark, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      udeg = degree_of(a.nindex, u);
      const bool join = seen != tag && udeg > 0;
      near = join && below;
      park = join && !below;
    }
  }
  frontier_emit_block(S.near, near, u, udeg, out, oc);
  se_park(S, park, u, nd, far, far_cnt);
}

// LDS of the team phase (shares the kernel's LDS with the emitter, which is idle
// meanwhile): the member's near share, and its own far pile by epoch parity.
struct SsspTeamLds {
  TeamShare<kShareCap> share;
  int far[2][kFarCap];
  int nfar[2];
  unsigned far_min[2];
  PhaseStop stop;
};

// Wave-collective: parks each lane's vertices u[q] (distance d[q]) with `park` in
// the member's far pile of `epoch`, past its capacity in the global one.
template <int kFly>
IG_DEV void team_park(const SsspArgs& a, SsspControl* ctl, SsspTeamLds& S, const bool (&park)[kFly],
                      const int (&u)[kFly], const int (&d)[kFly], int epoch)
{
  int mine = 0, least = kInf;
#pragma unroll
  for (int q = 0; q < kFly; q++) {
    if (park[q]) {
      mine++;
      least = min(least, d[q]);
    }
  }
  const int incl = wave_inclusive_scan(mine);
  const int all = wave_bcast(incl, kWave - 1);
  if (all == 0) return;
  const int p = epoch & 1;
  int slot = 0;
  if (lane_id() == 0) slot = atomicAdd(&S.nfar[p], all);
  slot = wave_bcast(slot, 0) + incl - mine;
#pragma unroll
  for (int q = 0; q < kFly; q++) {
    if (park[q]) {
      if (slot < kFarCap) S.far[p][slot] = u[q];
      else st_relaxed(&a.far[pile_of(epoch)][atomic_add_relaxed(&ctl->far_cnt[pile_of(epoch)].v, 1u)], u[q]);
      slot++;
    }
  }
  if (mine != 0) atomicMin(&S.far_min[p], static_cast<unsigned>(least));
}

// A team of workgroups (one, or up to kTeamMax) runs near iterations and
// splits alone while the near frontier's lists are short and few: team.hpp has
// the scheme.  To the grid the phase is one pass: entered with the near frontier
// in `in` (n vertices of the small queue, perhaps none), it leaves the frontier it
// reached (empty, or too large for the members) in `out` / `oc`, and everything
// parked in the global pile of the epoch it reached.  it, T and epoch are updated
// in place; they stay as they are where the members' shares do not all fit.
// *last gets the degree sum of the frontier before the one left.
//
// A near iteration is three dependent rounds of global accesses: the list
// entries, their weights and the vertices' own distances; the distance checks;
// and for those that pass, together, the minimum, the dedup exchange and the
// index pair (relax() has the reason).  Lists are walked as in the BFS kernel's
// team phase.  A split is one round and one more exchange: the members agree on
// the smallest parked distance, then each re-files its own pile (and its part of
// the global one); a pile holds a vertex once (farstamp), so marks are
// plain stores.  Roads of 1024^2, 2048^2 and 4096^2: 20.5, 49.5 and 215 -> 8.9,
// 24.9 and 65 ms a call (one workgroup took six dependent rounds and a binary
// search an iteration; wider frontiers and piles ran on the grid).
IG_DEV bool team_near(const SsspArgs& a, int& it, unsigned n, const Team& tm, int& T, int& epoch, int delta,
                      const FrontierQueues& in, const FrontierQueues& out, FrontierCounters* oc, SsspControl* ctl,
                      long long deadline, unsigned* last, SsspTeamLds& S)
{
  const int entry = epoch;  // (what others may still read, see split_waits)
  constexpr int kFly = 2;  // entries in flight per lane (3 and 4 spilled: 1024^2 road 8.9 ms a call, 9.3 and 11.9)
  const int t = static_cast<int>(threadIdx.x);
  TeamShare<kShareCap>& F = S.share;
  if (t == 0) {
    S.stop.clear();
    for (int p = 0; p < 2; p++) {
      S.nfar[p] = 0;
      S.far_min[p] = static_cast<unsigned>(kInf);
    }
  }
  unsigned entries = 0;
  int cn = share_load(F, it & 1, tm, static_cast<int>(n), a.nindex, [&](int i) { return ld_relaxed(&in.q[i]); },
                      &entries);
  TeamSum sum;
  if (!team_exchange(&ctl->team, kSlotEntry, tm, static_cast<unsigned>(it) + 1u, entries, 0u, &ctl->bar, deadline, F,
                     sum))
    return false;
  // (a share of more vertices than the LDS holds has more entries, too)
  if (sum.most > static_cast<unsigned>(kShareCap)) return true;
  for (;;) {
    if ((it & 63) == 0 && t == 0) S.stop.post(it, kernel_aborted(&ctl->bar, deadline));
    *last = sum.total;
    if (sum.total == 0u) {
      // near frontier empty: move the split and re-file the far piles
      const int p = epoch & 1;
      const int* gfar = a.far[pile_of(epoch)];
      const unsigned ng = ld_relaxed(&ctl->far_cnt[pile_of(epoch)].v);
      unsigned least = min(S.far_min[p], ld_relaxed(&ctl->far_min[pile_of(epoch)].v));
      if (!team_min(&ctl->team, tm, static_cast<unsigned>(it) + 1u, least, &ctl->bar, deadline, F, &least)) return false;
      if (least >= static_cast<unsigned>(kInf) || ng > static_cast<unsigned>(tm.size * kFarCap)) break;
      trace_level(&ctl->trace, it, ng + S.nfar[p], 0ull, 3);
      const int fmin = static_cast<int>(least);
      const int T_old = T;
      const long long Tn = static_cast<long long>(T > fmin ? T : fmin) + delta;
      T = Tn > kInf ? kInf : static_cast<int>(Tn);
      it++;
      epoch++;
      if (t == 0) {
        F.cnt[(it + 1) % 3] = 0ull;
        S.nfar[p ^ 1] = 0;
        S.far_min[p ^ 1] = static_cast<unsigned>(kInf);
        if (tm.rank == 0) {
          if (split_waits(entry, epoch - 1)) wait_others(&ctl->bar, tm, deadline);
          st_relaxed(&ctl->far_cnt[pile_cleared(epoch - 1)].v, 0u);
          st_relaxed(&ctl->far_min[pile_cleared(epoch - 1)].v, static_cast<unsigned>(kInf));
          ctl->epochs++;
        }
      }
      __syncthreads();
      const int own = min(S.nfar[p], kFarCap);
      const int part = (static_cast<int>(ng) - tm.rank + tm.size - 1) / tm.size;
      for (int base = 0; base < own + part; base += kSsspBlock) {
        const int i = base + t;
        bool near[1] = {false}, keep[1] = {false};
        int u[1] = {0}, du[1] = {0};
        IndexPair ip[1];
        if (i < own + part) {
          u[0] = i < own ? S.far[p][i] : ld_relaxed(&gfar[(i - own) * tm.size + tm.rank]);
          du[0] = ld_relaxed(&a.dist[u[0]]);
          ip[0] = index_pair(a.nindex, u[0]);
          near[0] = du[0] >= T_old && du[0] < T;
          keep[0] = du[0] >= T;
          if (near[0]) st_relaxed(&a.stamp[u[0]], it);
          if (keep[0]) st_relaxed(&a.farstamp[u[0]], epoch);
        }
        // what a full share cannot hold goes to the grid at once (and ends the phase)
        const bool over = share_append(F, it, near, u, ip);
        if (__ballot(over) != 0ull) frontier_emit(over, u[0], ip[0].end - ip[0].beg, out, oc);
        team_park(a, ctl, S, keep, u, du, epoch);
      }
    } else {
      trace_level(&ctl->trace, it, static_cast<unsigned>(cn), sum.total, 2);
      const int now = it & 1;
      it++;
      if (t == 0) F.cnt[(it + 1) % 3] = 0ull;
      int shift = 0;  // g = 1 << shift lanes per slot
      while (shift < 6 && (cn << (shift + 1)) <= kSsspBlock) shift++;
      const int sub = t & ((1 << shift) - 1);
      for (int i0 = 0; i0 < cn; i0 += kSsspBlock >> shift) {
        const int i = i0 + (t >> shift);
        const int beg = i < cn ? F.beg[now][i] : 0;
        const int end = i < cn ? beg + F.deg[now][i] : 0;
        const int dv = i < cn ? ld_relaxed(&a.dist[F.v[now][i]]) : 0;
        for (int e0 = beg + sub; __ballot(e0 < end) != 0ull; e0 += kFly << shift) {
          int u[kFly], nd[kFly];
          IndexPair ip[kFly];
          bool near[kFly], park[kFly];
#pragma unroll
          for (int q = 0; q < kFly; q++) {
            const int e = e0 + (q << shift);
            near[q] = e < end;
            u[q] = near[q] ? a.nlist[e] : 0;
            nd[q] = near[q] ? a.eweight[e] : 0;
          }
#pragma unroll
          for (int q = 0; q < kFly; q++) nd[q] += dv;
#pragma unroll
          for (int q = 0; q < kFly; q++) near[q] = near[q] && nd[q] < ld_relaxed(&a.dist[u[q]]);
#pragma unroll
          for (int q = 0; q < kFly; q++) {
            park[q] = false;
            if (near[q]) {
              const bool below = nd[q] < T;
              const int tag = below ? it : epoch;
              atomic_min_relaxed(&a.dist[u[q]], nd[q]);
              const int seen = __hip_atomic_exchange(below ? &a.stamp[u[q]] : &a.farstamp[u[q]], tag, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
              ip[q] = index_pair(a.nindex, u[q]);
              const bool join = seen != tag && ip[q].end > ip[q].beg;
              near[q] = join && below;
              park[q] = join && !below;
            }
          }
          share_append(F, it, near, u, ip);
          team_park(a, ctl, S, park, u, nd, epoch);
        }
      }
    }
    __syncthreads();
    if (S.stop.at(it - 1)) return false;  // (a turn is one near iteration or split)
    const unsigned long long c = F.cnt[it % 3];
    const bool full = (c & 0xffffffffull) > static_cast<unsigned long long>(kShareCap);
    cn = full ? kShareCap : static_cast<int>(c & 0xffffffffull);
    if (!team_exchange(&ctl->team, kSlotLevel + (it & 1), tm, static_cast<unsigned>(it),
                       full ? 0xffffu : static_cast<unsigned>(c >> 32), static_cast<unsigned>(cn), &ctl->bar, deadline,
                       F, sum))
      return false;
    if (sum.most == 0xffffu) break;
    if (share_uneven(tm, sum) && !share_deal(&ctl->team, it & 1, tm, static_cast<unsigned>(it), out.mq, a.nindex,
                                             &ctl->bar, deadline, F, cn, sum))
      return false;
    if (sum.most > (tm.size == 1 ? kSoloEntries : static_cast<unsigned>(kShareCap))) break;
  }
  // the rest of the frontier and the member's pile go to the grid
  const int own = min(S.nfar[epoch & 1], kFarCap);
  __syncthreads();
  if (t == 0 && own > 0) {
    S.nfar[0] = static_cast<int>(atomic_add_relaxed(&ctl->far_cnt[pile_of(epoch)].v, static_cast<unsigned>(own)));
    atomic_min_relaxed(&ctl->far_min[pile_of(epoch)].v, S.far_min[epoch & 1]);
  }
  __syncthreads();
  for (int i = t; i < own; i += kSsspBlock) st_relaxed(&a.far[pile_of(epoch)][S.nfar[0] + i], S.far[epoch & 1][i]);
  for (int base = 0; base < cn; base += kSsspBlock) {
    const int i = base + t;
    const int d = i < cn ? F.deg[it & 1][i] : 0;
    frontier_emit(d > 0, i < cn ? F.v[it & 1][i] : 0, d, out, oc);
  }
  return true;
}

// 6 waves per SIMD: three 512-thread workgroups per CU, the persistent grid's
// residency (at most 80 VGPRs)
__global__ __launch_bounds__(kSsspBlock) __attribute__((amdgpu_waves_per_eu(6, 8))) void sssp_kernel(SsspArgs a)
{
  __shared__ union {
    SsspEmit emit;
    SsspTeamLds small;
  } s_lds;
  SsspEmit& s_emit = s_lds.emit;
  SsspControl* ctl = a.ctl;
  if (!residency_barrier(&ctl->bar, a.start_ticks)) return;
  const long long deadline = now_ticks() + a.budget;
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  const int stride = gridDim.x * blockDim.x;
  const int lane = lane_id();
  if (tid == 0) ctl->trace.start = now_ticks();
  for (int i = tid; i < a.nodes; i += stride) {
    st_relaxed(&a.dist[i], (i == a.src) ? 0 : kInf);
    st_relaxed(&a.stamp[i], 0);
    st_relaxed(&a.farstamp[i], 0);
  }
  if (blockIdx.x == 0) {
    // delta: sampled mean weight x 32 / mean degree
    __shared__ long long s_wsum[kSsspBlock / kWave];
    __shared__ int s_ns[kSsspBlock / kWave];
    long long wsum = 0;
    int ns = 0;
    if (a.delta_hint <= 0 && a.edges > 0) {
      const int samples = a.edges < 4096 ? a.edges : 4096;
      for (int k = threadIdx.x; k < samples; k += blockDim.x) {
        const long long e = static_cast<long long>(k) * a.edges / samples;
        wsum += a.eweight[e];
        ns++;
      }
    }
    wsum = wave_sum(wsum);
    ns = wave_sum(ns);
    if (lane == 0) {
      s_wsum[threadIdx.x / kWave] = wsum;
      s_ns[threadIdx.x / kWave] = ns;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      int delta = a.delta_hint;
      if (delta <= 0) {
        long long ws = 0;
        int cnt = 0;
        for (int w = 0; w < kSsspBlock / kWave; w++) {
          ws += s_wsum[w];
          cnt += s_ns[w];
        }
        const double mean_w = cnt > 0 ? static_cast<double>(ws) / cnt : 1.0;
        const double mean_d = static_cast<double>(a.edges) / a.nodes;
        double d = mean_w * 32.0 / (mean_d > 1.0 ? mean_d : 1.0);
        delta = d < 1.0 ? 1 : (d > 1e9 ? 1000000000 : static_cast<int>(d));
      }
      st_relaxed(&ctl->delta, delta);
      for (int k = 0; k < 3; k++) st_relaxed(&ctl->far_min[k].v, static_cast<unsigned>(kInf));
    }
    __syncthreads();
    if (threadIdx.x < kWave) {
      const int deg = degree_of(a.nindex, a.src);
      frontier_emit(threadIdx.x == 0 && deg > 0, a.src, deg, a.fq[0], &ctl->cnt[0]);
    }
  }
  if (!grid_barrier<true>(&ctl->bar, deadline)) {
    if (tid == 0) ctl->status = 1;
    return;
  }
  const int delta = ld_relaxed(&ctl->delta);
  int T = delta;  // split: near holds distances < T
  int epoch = 1;  // far pile generation (farstamp value); far[pile_of(epoch)] is current
  int it = 0;     // near iterations and splits (stamp values start at 1)
  int R = 0;      // pass: counters rotate and queues alternate by it
  int declined = -1;           // iteration that a team has left to the grid
  unsigned long long prev = 0;  // degree sum of the frontier before
  for (;;) {
    FrontierCounters* ic = &ctl->cnt[R % 3];
    const unsigned n = ld_relaxed(&ic->n);
    const unsigned nm = ld_relaxed(&ic->nm);
    const unsigned long long hp = ld_relaxed(&ic->hpack);
    const unsigned nh = huge_count(hp), nch = huge_chunks(hp);
    FrontierCounters* oc = &ctl->cnt[(R + 1) % 3];
    const FrontierQueues& in = a.fq[R & 1];
    const FrontierQueues& out = a.fq[(R + 1) & 1];
    if (tid == 0) counters_clear(&ctl->cnt[(R + 2) % 3]);
    int* far = a.far[pile_of(epoch)];
    unsigned* far_cnt = &ctl->far_cnt[pile_of(epoch)].v;
    unsigned* far_min = &ctl->far_min[pile_of(epoch)].v;
    const bool split = static_cast<unsigned long long>(n) + nm + nh == 0;
    const unsigned long long m = ld_relaxed(&ic->m);
    const unsigned nfar = split ? ld_relaxed(far_cnt) : 0u;
    if (split && nfar == 0) break;
    int team = 0;  // workgroups of a team phase, 0: a grid pass
    if (a.allow_small && declined != it && nm == 0 && nh == 0) {
      const int limit = team_limit();
      if (split) team = nfar <= static_cast<unsigned>(kFarCap) ? 1 : 0;
      else if (m <= kSoloEntries) team = 1;
      else if (m <= static_cast<unsigned long long>(limit) * kShareEntries && m <= 2ull * prev) team = limit;
    }
    prev = m;
    trace_level(&ctl->trace, it, split ? nfar : n + nm + nh, split ? 0ull : m, split ? 3 : (team != 0 ? 2 : 0));
    if (team != 0) {
      // the workgroups outside the team wait at the next barrier
      const Team tm = make_team(team);
      if (tm.rank >= 0) {
        int it2 = it, T2 = T, epoch2 = epoch;
        unsigned last = 0;
        // (false: the kernel's abort mark is set, and the barrier below says so
        // to the whole workgroup; a return here spilled 42 registers instead of 15)
        const bool ok = team_near(a, it2, n, tm, T2, epoch2, delta, in, out, oc, ctl, deadline, &last, s_lds.small);
        if (ok && tm.rank == 0 && threadIdx.x == 0) {
          st_relaxed(&ctl->base.of(R).it, it2);
          st_relaxed(&ctl->base.of(R).split, T2);
          st_relaxed(&ctl->base.of(R).epoch, epoch2);
          st_relaxed(&ctl->base.of(R).last_m, last);
          ctl->small_iters += it2 - it;
        }
      }
      if (!grid_barrier<true>(&ctl->bar, deadline)) {
        if (tid == 0) ctl->status = 1;
        return;
      }
      const int it2 = ld_relaxed(&ctl->base.of(R).it);
      if (it2 == it) {  // an uneven frontier: this pass goes to the grid
        declined = it;
        continue;
      }
      it = it2;
      T = ld_relaxed(&ctl->base.of(R).split);
      epoch = ld_relaxed(&ctl->base.of(R).epoch);
      prev = ld_relaxed(&ctl->base.of(R).last_m);
      R++;
      continue;
    }
    if (split) {
      // near frontier empty: move the split and re-file the far pile
      const unsigned nf = nfar;
      const int fmin = static_cast<int>(ld_relaxed(far_min));
      const int T_old = T;
      const long long Tn = static_cast<long long>(T > fmin ? T : fmin) + delta;
      T = Tn > kInf ? kInf : static_cast<int>(Tn);
      it++;
      const int nepoch = epoch + 1;
      int* nfar = a.far[pile_of(nepoch)];
      unsigned* nfar_cnt = &ctl->far_cnt[pile_of(nepoch)].v;
      unsigned* nfar_min = &ctl->far_min[pile_of(nepoch)].v;
      if (tid == 0) {
        // (consumed by the previous split, one barrier ago)
        st_relaxed(&ctl->far_cnt[pile_cleared(epoch)].v, 0u);
        st_relaxed(&ctl->far_min[pile_cleared(epoch)].v, static_cast<unsigned>(kInf));
      }
      se_reset(s_emit);
      for (unsigned base = blockIdx.x * blockDim.x; base < nf; base += stride) {
        const unsigned i = base + threadIdx.x;
        bool to_near = false, keep = false;
        int u = 0, du = 0, udeg = 0;
        if (i < nf) {
          u = ld_relaxed(&far[i]);
          du = ld_relaxed(&a.dist[u]);
          if (du >= T_old) {
            if (du < T) {
              to_near = __hip_atomic_exchange(&a.stamp[u], it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != it;
              if (to_near) udeg = degree_of(a.nindex, u);
            } else {
              keep = __hip_atomic_exchange(&a.farstamp[u], nepoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != nepoch;
            }
          }
        }
        frontier_emit_block(s_emit.near, to_near, u, udeg, out, oc);
        se_park(s_emit, keep, u, du, nfar, nfar_cnt);
      }
      se_flush(s_emit, out, oc, nfar, nfar_cnt, nfar_min);
      if (tid == 0) ctl->epochs++;
      epoch = nepoch;
    } else {
      it++;
      se_reset(s_emit);
      auto visit = [&](int v, int e, bool active) {
        const int dv = active ? ld_relaxed(&a.dist[v]) : 0;
        relax(a, dv, e, active, T, it, epoch, far, far_cnt, s_emit, out, oc);
      };
      expand_huge(in, nh, nch, a.nindex, visit);
      expand_mid(in, nm, a.nindex, visit);
      const unsigned avg = nm + nh == 0 ? static_cast<unsigned>(m / n) : 16u;
      expand_small(in.q, n, a.nindex, visit, small_share(n, avg));
      se_flush(s_emit, out, oc, far, far_cnt, far_min);
    }
    if (!grid_barrier<true>(&ctl->bar, deadline)) {
      if (tid == 0) ctl->status = 1;
      return;
    }
    R++;
  }
  if (tid == 0) ctl->iterations = it;
}

}  // namespace

size_t sssp_workspace_bytes(int nodes)
{
  const size_t v = static_cast<size_t>(nodes);
  return Carver::round(sizeof(SsspControl)) + 13 * Carver::round(v * 4) + 4096;
}

int sssp_run(indigo_ctx* ctx, int nodes, int edges, const int* nindex, const int* nlist, const int* eweight, int src,
             int* dist)
{
  Carver cv(ctx->ws);
  SsspArgs a{};
  a.ctl = cv.take<SsspControl>(1);
  for (int k = 0; k < 2; k++) {
    a.fq[k].q = cv.take<int>(nodes);
    a.fq[k].mq = cv.take<int>(nodes);
    a.fq[k].hq = cv.take<int>(nodes);
    a.fq[k].hoff = cv.take<unsigned>(nodes);
  }
  for (int k = 0; k < 3; k++) a.far[k] = cv.take<int>(nodes);
  a.stamp = cv.take<int>(nodes);
  a.farstamp = cv.take<int>(nodes);
  a.nodes = nodes;
  a.edges = edges;
  a.src = src;
  a.delta_hint = ctx->hints[INDIGO_HINT_SSSP_DELTA];
  a.allow_small = ctx->hints[INDIGO_HINT_SMALL_FRONTIER] != 1;
  a.nindex = nindex;
  a.nlist = nlist;
  a.eweight = eweight;
  a.dist = dist;
  a.budget = budget_ticks(ctx);
  a.start_ticks = residency_ticks(ctx);
  IG_TRY(zero_async(ctx, a.ctl, sizeof(SsspControl)));
  void* args[] = {&a};
  IG_TRY(coop_launch(ctx, reinterpret_cast<const void*>(sssp_kernel), kSsspBlock, 0, args, 0, nullptr, "sssp_kernel"));
  return INDIGO_OK;
}

int sssp_collect(indigo_ctx* ctx, int* iterations, int* epochs)
{
  Carver cv(ctx->ws);
  SsspControl* ctl = cv.take<SsspControl>(1);
  IG_TRY(ensure_host_pinned(ctx, sizeof(SsspControl)));
  SsspControl* h = static_cast<SsspControl*>(ctx->host_pinned);
  IG_HIP_TRY(hipMemcpyAsync(h, ctl, sizeof(SsspControl), hipMemcpyDeviceToHost, ctx->stream));
  IG_HIP_TRY(hipStreamSynchronize(ctx->stream));
  IG_TRY(check_abort(ctx, reinterpret_cast<const void*>(sssp_kernel), h->bar.abort.v, "sssp"));
  if (h->status != 0) return set_error(INDIGO_ERR_TIMEOUT, "sssp: persistent kernel stopped (status %d)", h->status);
  if (iterations) *iterations = h->iterations;
  if (epochs) *epochs = h->epochs;
  store_trace(ctx, h->trace);
  return INDIGO_OK;
}

}  // namespace indigo
