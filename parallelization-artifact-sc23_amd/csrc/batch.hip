// Batched engine: many graphs and many sources per graph in one persistent
// launch (MI355X, gfx950).
//
// Every query becomes a task: multi-source BFS (up to 64 sources), multi-
// source SSSP (up to 32), CC, MIS or PageRank on one graph.  The host sorts
// tasks by size (largest first) into a device-side queue; one persistent
// kernel, sized to co-residency and checked by a residency barrier, serves
// it.
//
// Gangs.  A task runs on a gang of k workgroups, k = the task's CSR entries
// / 2^18 rounded up to a power of two: small graphs take one workgroup and
// synchronise with __syncthreads only, large ones a gang with its own bounded
// barrier.  Where that leaves workgroups of the grid without a task, the tasks
// that would finish last take them (widen_gangs).  The cap depends on how much
// work a barrier separates: 256 for the dense sweeps of PR, CC and MIS, 128 for
// BFS, 64 for SSSP's many short rounds (256 of idle workgroups), and 16 for BFS
// on sparse graphs (average degree below 6), which may have thousands of
// levels, each bound by barrier latency.  A free workgroup joins the first task in queue
// order that still has a free slot (one atomic on the task's `joined`
// counter); the gang starts when all k members have arrived.  Because every
// workgroup is resident and gangs are filled strictly in queue order, a gang
// only ever waits for workgroups that are busy with earlier tasks, so
// formation cannot deadlock.
//
// Load balance inside a task.  Sweeps give each wave 64 consecutive vertices
// (or queue entries) and walk their lists 64 entries per step with the
// in-wave balancer.  Lists of kHeavyDeg entries or more would tie a wave up
// (R-MAT hubs reach 10^5 entries), so each task first lists its heavy
// vertices as kItem-entry items that all waves of the gang share; sweeps
// skip heavy lists and a second loop walks the items.
//
// Memory discipline (as the coherent-mode persistent kernels): data one
// thread writes and another reads within a task, or that two threads write,
// goes through device-scope relaxed loads / stores / atomics (the eight XCDs'
// L2 caches are not coherent for plain accesses, and these barriers do not
// write them back), and each barrier first drains the wave's memory
// operations; barriers are relaxed counters.  Plain stores remain only for
// slab entries written exactly once.
//
// Algorithms (same results as the single-query kernels and the reference):
//   BFS : level-synchronous and direction-optimising over 64-bit masks:
//         frontier[v] holds the sources whose BFS reached v at the previous
//         level, and the frontier vertices are also kept in a queue.  While
//         the frontier's lists hold fewer than E / 14 entries it pushes:
//         each frontier vertex ORs its mask, minus the bits a neighbour has
//         seen, into the neighbour's next mask, and the first push into a
//         vertex queues it.  Otherwise it pulls: every vertex with sources
//         still missing ORs its neighbours' frontier masks.  A second phase
//         turns the next masks into the new frontier and writes the level
//         into the slab rows of the new bits.  A level costs its edge work plus
//         two barriers: the gang's, or the workgroup's for levels of at most kNarrow
//         entries, which member 0 runs alone.
//   SSSP: Bellman-Ford driven by a queue of active vertices over vertex-major
//         rows of distances, with a mask of the sources that are active at a vertex;
//         lists are taken in blocks of 64 entries, whose (entry, source) pairs are
//         relaxed by atomicMin, and a vertex is queued for the next round when its
//         distance for some source drops.  Sources go through in passes where
//         their rows do not fit the memory.  Narrow rounds are member 0's, too.
//   CC  : union-find hooking the larger root under the smaller (labels =
//         component minima), then flattening; graphs of average degree 8 or
//         more link in Afforest order and skip the giant component's lists.
//   MIS : the greedy fixed point in descending (hash(v + 712313887), v)
//         order; rounds of decisions in place, as the single-query kernel's (a
//         vertex joins when its larger neighbours are all excluded, and is
//         excluded once one of them is included).  A heavy vertex's items
//         raise per-vertex flags, by which it is decided in the next round.
//         Deferring a decision changes no result: a vertex decides only once
//         every larger undecided neighbour has, as in the greedy order.
//   PR  : the Jacobi recurrence of the single-query kernel (FP32 scores,
//         Neumaier-compensated gathers: one lane per list of fewer than
//         kPrLaneDeg entries in entry order, eight lanes or a wave per longer one,
//         per-item partials combined in item order for heavy lists),
//         stopping when the FP64 L1 change is <= 1e-4 or after 100 sweeps;
//         every gang member adds the members' FP64 partials in the same
//         order, so all take the same decision.
#include "batch.hpp"

#include <algorithm>
#include <climits>
#include <cstring>
#include <queue>
#include <utility>
#include <vector>

#include "device_common.hpp"
#include "emit.hpp"
#include "gather.hpp"
#include "mis_decide.hpp"
#include "unionfind.hpp"

namespace indigo {

namespace {

constexpr int kBatchBlock = 512;
constexpr int kBatchWaves = kBatchBlock / kWave;
constexpr int kMaxGang = INDIGO_MAX_GANG;
constexpr int kGangShift = 18;   // CSR entries per gang member
constexpr int kWidenEntries = 4096;  // CSR entries per member of a widened gang (widen_floor)
constexpr int kHeavyDeg = 1024;  // lists this long are split into items
constexpr int kItem = 1024;      // entries per item
constexpr int kMisWaveList = 64;   // MIS: lists finished by a whole wave
constexpr int kCcSample = 2;      // CC: neighbours linked per vertex before the giant root is chosen
constexpr int kCcDepth = 2;       // CC: hops beyond which a find stores the root (100 graphs: 5.1 / 4.7 / 4.7 / 7.6 ms at 5 / 2 / 1 / 0)
constexpr int kCcSamples = 256;   // CC: vertices sampled to choose it
constexpr int kCcAfforestMin = 4096;  // CC: smallest graph that takes the Afforest order
constexpr int kBatchQueue = 2048;  // BFS, SSSP: appends that a workgroup buffers per round
constexpr float kDamp = 0.85f;

struct alignas(128) GangState {
  unsigned long long mf[4];  // BFS: degree sums of the queued frontiers, rotated by level
  unsigned joined;           // members that took a slot (grows past the gang size)
  unsigned arrive;           // barrier arrivals of the current generation
  unsigned gen;              // barrier generation
  unsigned flag[3];          // per-round "something changed" flags, triple-buffered
  unsigned qn[4];            // frontier queue sizes, rotated by level / round
  unsigned nitems;           // heavy-list items
  unsigned grp[8];           // barrier arrivals per rank group (gangs above 16)
  unsigned pad[5];
};

struct BatchTask {
  int alg, gang, nodes, edges;
  const int* nindex;
  const int* nlist;
  const int* eweight;
  int* out;
  void* scratch;  // per algorithm, see scratch_bytes
  int2* items;    // heavy-list items (vertex, first entry)
  int item;       // lists of this many entries or more are split into items of as many
  int nsrc;
  int rows;       // SSSP: sources of one pass, a power of two (scratch_bytes)
  int src[INDIGO_MAX_BFS_SOURCES];
};

struct alignas(128) BatchControl {
  GridBarrier bar;
  unsigned head;  // first task that may still have a free slot
  unsigned pad[31];
};

struct Team {
  int rank, size;
  GangState* gs;
  GridBarrier* gb;
  long long deadline;
};

// Gang barrier (bounded).  Size 1: the workgroup barrier suffices; up to 64
// members count on one counter, larger gangs first on a counter per rank
// group (rank mod 8), then the groups' last arrivals on the shared one.
IG_DEV bool team_sync(const Team& tm)
{
  __shared__ int s_ok;
  wave_drain();
  __syncthreads();
  if (threadIdx.x == 0) {
    int ok = 1;
    if (tm.size > 1) {
      const unsigned gen0 = ld_relaxed(&tm.gs->gen);
      wave_drain();
      bool last = false;
      if (tm.size <= 64) {
        last = atomic_add_relaxed(&tm.gs->arrive, 1u) == static_cast<unsigned>(tm.size) - 1u;
      } else {
        const unsigned g = static_cast<unsigned>(tm.rank) & 7u;
        const unsigned gsize = (static_cast<unsigned>(tm.size) - g + 7u) >> 3;  // ranks r < size with r % 8 == g
        if (atomic_add_relaxed(&tm.gs->grp[g], 1u) == gsize - 1u) {
          st_relaxed(&tm.gs->grp[g], 0u);
          wave_drain();
          last = atomic_add_relaxed(&tm.gs->arrive, 1u) == 7u;
        }
      }
      if (last) {
        st_relaxed(&tm.gs->arrive, 0u);
        wave_drain();
        st_relaxed(&tm.gs->gen, gen0 + 1u);
      } else {
        int backoff = 1;
        while (ld_relaxed(&tm.gs->gen) == gen0) {
          if (ld_relaxed(&tm.gb->abort.v) != 0u) break;
          if (now_ticks() > tm.deadline) {
            unsigned expected = 0u;
            __hip_atomic_compare_exchange_strong(&tm.gb->abort.v, &expected, kAbortTimeout, __ATOMIC_RELAXED,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
          }
          for (int k = 0; k < backoff; k++) __builtin_amdgcn_s_sleep(1);
          backoff = backoff < 8 ? backoff * 2 : 8;  // short polls: gangs wait a few microseconds per level
        }
      }
    } else if (now_ticks() > tm.deadline) {
      unsigned expected = 0u;
      __hip_atomic_compare_exchange_strong(&tm.gb->abort.v, &expected, kAbortTimeout, __ATOMIC_RELAXED,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (ld_relaxed(&tm.gb->abort.v) != 0u) ok = 0;
    s_ok = ok;
  }
  __syncthreads();
  return s_ok != 0;
}

IG_DEV void wave_lds_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// SSSP: log2 of a vertex's distances in the vertex-major rows.
__host__ __device__ inline int sssp_row_shift(int nsrc)
{
  int s = 0;
  while ((1 << s) < nsrc) s++;
  return s;
}

IG_DEV bool heavy(int deg) { return deg >= kHeavyDeg; }

// Wave-collective: walks the CSR entries of the vertex `v` of each lane with
// `active` and a list shorter than kHeavyDeg, 64 per step; f(o, e, valid)
// gets the owner lane o and the entry e, with all lanes converged.
template <typename F>
IG_DEV void wave_entries_of(int v, bool active, const int* __restrict__ nindex, F&& f)
{
  const int lane = lane_id();
  const int b = active ? nindex[v] : 0;
  const int l = active ? nindex[v + 1] - b : 0;
  const int len = heavy(l) ? 0 : l;
  const int incl = wave_inclusive_scan(len);
  const int total = wave_bcast(incl, kWave - 1);
  const int shift = b - (incl - len);
  for (int base = 0; base < total; base += kWave) {
    const int k = base + lane;
    const int o = min(wave_owner(incl, k), kWave - 1);
    const int e = wave_shfl(shift, o) + k;
    f(o, e, k < total);
  }
}

// The team's share of 64-vertex chunks: chunk c for c = first, first + step, ...
struct Chunks {
  int first, step, count;
};

IG_DEV Chunks team_chunks(const Team& tm, int n)
{
  return Chunks{tm.rank * kBatchWaves + static_cast<int>(threadIdx.x) / kWave, tm.size * kBatchWaves,
                (n + kWave - 1) / kWave};
}

// Wave-collective: f(v, e_begin, e_end, item) for the team's share of the
// heavy items (one item per wave at a time).
template <typename F>
IG_DEV void for_items(const BatchTask& T, const Team& tm, int nitems, F&& f)
{
  for (int i = tm.rank * kBatchWaves + static_cast<int>(threadIdx.x) / kWave; i < nitems;
       i += tm.size * kBatchWaves) {
    const int v = ld_relaxed(&T.items[i].x), eb = ld_relaxed(&T.items[i].y);
    f(v, eb, min(eb + kItem, T.nindex[v + 1]), i);
  }
}

// Gang-collective, once per task: lists the heavy vertices' items.
IG_DEV bool build_items(const BatchTask& T, const Team& tm, int* nitems)
{
  const int lane = lane_id();
  const Chunks ch = team_chunks(tm, T.nodes);
  for (int c = ch.first; c < ch.count; c += ch.step) {
    const int v = c * kWave + lane;
    const int b = v < T.nodes ? T.nindex[v] : 0;
    const int deg = v < T.nodes ? T.nindex[v + 1] - b : 0;
    const int n = deg >= T.item ? (deg + T.item - 1) / T.item : 0;
    const int incl = wave_inclusive_scan(n);
    const int total = wave_bcast(incl, kWave - 1);
    if (total == 0) continue;
    unsigned base = 0;
    if (lane == 0) base = atomic_add_relaxed(&tm.gs->nitems, static_cast<unsigned>(total));
    base = static_cast<unsigned>(wave_shfl(static_cast<int>(base), 0));
    for (int j = 0; j < n; j++) {
      const unsigned slot = base + static_cast<unsigned>(incl - n + j);
      st_relaxed(&T.items[slot].x, v);
      st_relaxed(&T.items[slot].y, b + j * T.item);
    }
  }
  if (!team_sync(tm)) return false;
  *nitems = static_cast<int>(ld_relaxed(&tm.gs->nitems));
  return true;
}

IG_DEV void set_flag(unsigned* flag, bool any)
{
  if (__ballot(any) != 0ull && lane_id() == 0) st_relaxed(flag, 1u);
}

// Or of the 64 lanes' words, the same in all (all lanes must be active): the steps of
// wave_inclusive_scan, whose last lane has the whole.
IG_DEV unsigned wave_or32(unsigned x)
{
  int y = static_cast<int>(x);
  y |= __builtin_amdgcn_update_dpp(0, y, 0x111, 0xf, 0xf, false);  // row_shr:1
  y |= __builtin_amdgcn_update_dpp(0, y, 0x112, 0xf, 0xf, false);  // row_shr:2
  y |= __builtin_amdgcn_update_dpp(0, y, 0x114, 0xf, 0xf, false);  // row_shr:4
  y |= __builtin_amdgcn_update_dpp(0, y, 0x118, 0xf, 0xf, false);  // row_shr:8
  y |= __builtin_amdgcn_update_dpp(0, y, 0x142, 0xa, 0xf, false);  // row_bcast:15
  y |= __builtin_amdgcn_update_dpp(0, y, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return static_cast<unsigned>(wave_bcast(y, kWave - 1));
}

IG_DEV unsigned long long wave_or(unsigned long long x)
{
  return static_cast<unsigned long long>(wave_or32(static_cast<unsigned>(x >> 32))) << 32 |
         wave_or32(static_cast<unsigned>(x));
}

// Wave-collective: walks the lists as wave_entries_of does, kFly entries per lane
// at a time, and hands over the owner lanes, the neighbours and which of them are
// there: f(o, u, on), arrays of kFly.
constexpr int kFly = 2;
// BFS: entries of a narrow level, for one member (one step of 64 per wave; below kHeavyDeg);
// SSSP: vertices of a narrow round, left again above four times as many.
constexpr unsigned long long kNarrow = 512;
constexpr int kNarrowQueue = 32;
constexpr int kLaneFly = 2;                  // SSSP: sources of an entry that its lane takes alone
constexpr int kGroupFly = 2;                 // SSSP: steps in flight that take a group of lanes per entry

template <typename F>
IG_DEV void wave_neighbours_of(int v, bool active, const BatchTask& T, F&& f)
{
  const int lane = lane_id();
  const int b = active ? T.nindex[v] : 0;
  const int l = active ? T.nindex[v + 1] - b : 0;
  const int len = heavy(l) ? 0 : l;
  const int incl = wave_inclusive_scan(len);
  const int total = wave_bcast(incl, kWave - 1);
  const int shift = b - (incl - len);
  for (int base = 0; base < total; base += kFly * kWave) {
    int o[kFly], u[kFly];
    bool on[kFly];
#pragma unroll
    for (int q = 0; q < kFly; q++) {
      const int k = base + q * kWave + lane;
      on[q] = k < total;
      o[q] = min(wave_owner(incl, k), kWave - 1);
      const int e = wave_shfl(shift, o[q]) + k;
      u[q] = on[q] ? T.nlist[e] : 0;
    }
    f(o, u, on);
  }
}

// Wave-collective: f as above for the entries [eb, ee) of one list (o is 0).
template <typename F>
IG_DEV void item_neighbours(int eb, int ee, const BatchTask& T, F&& f)
{
  for (int e0 = eb; e0 < ee; e0 += kFly * kWave) {
    int o[kFly], u[kFly];
    bool on[kFly];
#pragma unroll
    for (int q = 0; q < kFly; q++) {
      const int e = e0 + q * kWave + lane_id();
      on[q] = e < ee;
      o[q] = 0;
      u[q] = on[q] ? T.nlist[e] : 0;
    }
    f(o, u, on);
  }
}

// ---- multi-source BFS -------------------------------------------------------
// Wave-collective: level to the slab rows of each lane's sources m, entry v.  The
// wave takes a row at a time, so the stores of neighbouring vertices (pulls queue
// them in order) go out together.
IG_DEV void write_rows(const BatchTask& T, unsigned long long m, int v, int level)
{
  // ... and few sources per vertex each lane its own: a path's frontier of 128 vertices for
  // 64 sources cost a BFS 64 turns of the wave a level (10.5 -> 7.8 us).
  unsigned long long rows = wave_or(m);
  const int bits = wave_bcast(wave_inclusive_scan(__popcll(m)), kWave - 1);
  if (4 * bits >= kWave * __popcll(rows)) {
    for (; rows != 0ull; rows &= rows - 1ull) {
      const int i = __ffsll(static_cast<long long>(rows)) - 1;
      if (m >> i & 1ull) T.out[static_cast<size_t>(i) * T.nodes + v] = level;
    }
  } else {
    for (; m != 0ull; m &= m - 1ull)
      T.out[static_cast<size_t>(__ffsll(static_cast<long long>(m)) - 1) * T.nodes + v] = level;
  }
}

// Bound by the latency of its steps (list entry, mask, append).  The appends of a
// level and their degree sum are gathered in LDS and registers instead of two
// atomics and a 64-bit wave sum a step, two entries per lane are in flight and the
// levels are written a row at a time: 100 graphs of 64 sources 32.6 -> 27.2 ms.
// Gang-collective over the members of w: level lvl from its frontier of ncur vertices with
// mcur entries; *count and *entries get the next one's, which each member has read when
// the level ends.
IG_DEV bool bfs_level(const BatchTask& T, const Team& w, int lvl, int nitems, unsigned long long all, int ncur,
                      unsigned long long mcur, int* count, unsigned long long* entries,
                      unsigned long long (*s_acc)[kWave], BlockQueue<kBatchQueue>& s_next, BlockSum& s_mf)
{
  const int V = T.nodes;
  const int lane = lane_id();
  const int wid = threadIdx.x / kWave;
  const size_t Vs = static_cast<size_t>(V);
  unsigned long long* seen = static_cast<unsigned long long*>(T.scratch);
  unsigned long long* fr[2] = {seen + Vs, seen + 2 * Vs};  // frontier masks by level parity
  unsigned long long* nxt = seen + 3 * Vs;                 // next-level masks
  int* queue[2] = {reinterpret_cast<int*>(seen + 4 * Vs), reinterpret_cast<int*>(seen + 4 * Vs) + V};
  unsigned* qn = w.gs->qn;
  unsigned long long* mf = w.gs->mf;
  const Chunks ch = team_chunks(w, V);
  const unsigned long long* cur = fr[(lvl - 1) & 1];
  unsigned long long* nfr = fr[lvl & 1];
  const int* qcur = queue[(lvl - 1) & 1];
  int* qnext = queue[lvl & 1];
  unsigned* ncount = &qn[lvl & 3];
  unsigned long long* nmf = &mf[lvl & 3];
  if (w.rank == 0 && threadIdx.x == 0) {
    st_relaxed(&qn[(lvl + 1) & 3], 0u);
    st_relaxed(&mf[(lvl + 1) & 3], 0ull);
  }
  // Narrow levels append straight to the queue: the buffer's four workgroup barriers cost
  // them more than its atomics save (path of 2^15 vertices, one workgroup: 2.8 -> 2.6 us a level).
  const bool direct = mcur <= kNarrow * static_cast<unsigned long long>(w.size);
  if (!direct) {
    if (threadIdx.x == 0) s_mf.v = 0ull;
    bq_reset(s_next);
  }
  int dsum = 0;  // degrees of what this lane appends
  auto append = [&](bool first, int u) {
    if (first) dsum += T.nindex[u + 1] - T.nindex[u];
    if (direct) wave_append(first, u, qnext, ncount);
    else bq_append(s_next, first, u, qnext, ncount);
  };
  if (mcur * 14ull < static_cast<unsigned long long>(T.edges)) {
    // push from the frontier queue
    const int nq = (ncur + kWave - 1) / kWave;
    auto push = [&](const unsigned long long (&m)[kFly], const int (&u)[kFly], const bool (&on)[kFly]) {
      unsigned long long add[kFly];
      bool first[kFly];
#pragma unroll
      for (int q = 0; q < kFly; q++) add[q] = on[q] ? m[q] & ~ld_relaxed(&seen[u[q]]) : 0ull;
#pragma unroll
      for (int q = 0; q < kFly; q++)
        first[q] = add[q] != 0ull && __hip_atomic_fetch_or(&nxt[u[q]], add[q], __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_AGENT) == 0ull;
#pragma unroll
      for (int q = 0; q < kFly; q++) append(first[q], u[q]);
    };
    for (int c = ch.first; c < nq; c += ch.step) {
      const int k = c * kWave + lane;
      const bool act = k < ncur;
      const int v = act ? ld_relaxed(&qcur[k]) : 0;
      const unsigned long long m = act ? ld_relaxed(&cur[v]) : 0ull;
      wave_neighbours_of(v, act, T, [&](const int (&o)[kFly], const int (&u)[kFly], const bool (&on)[kFly]) {
        unsigned long long om[kFly];
#pragma unroll
        for (int q = 0; q < kFly; q++) om[q] = __shfl(m, o[q], kWave);
        push(om, u, on);
      });
    }
    // (a heavy vertex alone has kHeavyDeg entries)
    if (mcur >= static_cast<unsigned long long>(kHeavyDeg)) for_items(T, w, nitems, [&](int v, int eb, int ee, int) {
      const unsigned long long m = ld_relaxed(&cur[v]);
      if (m == 0ull) return;
      item_neighbours(eb, ee, T, [&](const int (&)[kFly], const int (&u)[kFly], const bool (&on)[kFly]) {
        unsigned long long om[kFly];
#pragma unroll
        for (int q = 0; q < kFly; q++) om[q] = m;
        push(om, u, on);
      });
    });
  } else {
    // pull: every vertex with sources still missing
    for (int c = ch.first; c < ch.count; c += ch.step) {
      const int v = c * kWave + lane;
      const unsigned long long sv = v < V ? ld_relaxed(&seen[v]) : all;
      const unsigned long long missing = all & ~sv;
      s_acc[wid][lane] = 0ull;
      wave_lds_sync();
      wave_neighbours_of(v, missing != 0ull, T, [&](const int (&o)[kFly], const int (&u)[kFly], const bool (&on)[kFly]) {
        unsigned long long m[kFly];
#pragma unroll
        for (int q = 0; q < kFly; q++) m[q] = on[q] ? ld_relaxed(&cur[u[q]]) : 0ull;
#pragma unroll
        for (int q = 0; q < kFly; q++)
          if (m[q] != 0ull) atomicOr(&s_acc[wid][o[q]], m[q]);
      });
      wave_lds_sync();
      const unsigned long long nb = s_acc[wid][lane] & missing;
      if (nb != 0ull) st_relaxed(&nxt[v], nb);
      append(nb != 0ull, v);
    }
    for_items(T, w, nitems, [&](int v, int eb, int ee, int) {
      const unsigned long long missing = all & ~ld_relaxed(&seen[v]);
      if (missing == 0ull) return;
      unsigned long long acc = 0ull;
      item_neighbours(eb, ee, T, [&](const int (&)[kFly], const int (&u)[kFly], const bool (&on)[kFly]) {
        unsigned long long m[kFly];
#pragma unroll
        for (int q = 0; q < kFly; q++) m[q] = on[q] ? ld_relaxed(&cur[u[q]]) : 0ull;
#pragma unroll
        for (int q = 0; q < kFly; q++) acc |= m[q];
      });
      const unsigned long long nb = wave_or(acc) & missing;
      bool first = false;
      if (nb != 0ull && lane == 0)
        first = __hip_atomic_fetch_or(&nxt[v], nb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0ull;
      append(first, v);
    });
  }
  // (a vertex is appended once a level: the sum stays below 2^31)
  const int degrees = wave_bcast(wave_inclusive_scan(dsum), kWave - 1);
  if (direct) {
    if (degrees != 0 && lane == 0) atomic_add_relaxed(nmf, static_cast<unsigned long long>(degrees));
  } else {
    if (degrees != 0 && lane == 0) atomicAdd(&s_mf.v, static_cast<unsigned long long>(degrees));
    bq_flush<false>(s_next, qnext, ncount);
    if (threadIdx.x == 0 && s_mf.v != 0ull) atomic_add_relaxed(nmf, s_mf.v);
  }
  if (!team_sync(w)) return false;
  // the new frontier: masks, seen bits and levels; the old frontier's masks
  // are cleared (that buffer holds the next level's frontier)
  const int nnext = static_cast<int>(ld_relaxed(ncount));
  *count = nnext;
  *entries = ld_relaxed(nmf);
  for (int k = w.rank * kBatchBlock + static_cast<int>(threadIdx.x); k < ncur; k += w.size * kBatchBlock)
    st_relaxed(&fr[(lvl - 1) & 1][ld_relaxed(&qcur[k])], 0ull);
  for (int c = ch.first; c * kWave < nnext; c += ch.step) {
    const int k = c * kWave + lane;
    const int u = k < nnext ? ld_relaxed(&qnext[k]) : 0;
    unsigned long long nb = 0ull;
    if (k < nnext) {
      const unsigned long long sv = ld_relaxed(&seen[u]);
      nb = ld_relaxed(&nxt[u]) & ~sv;
      st_relaxed(&nxt[u], 0ull);
      st_relaxed(&seen[u], sv | nb);
      st_relaxed(&nfr[u], nb);
    }
    write_rows(T, nb, u, lvl);
  }
  return team_sync(w);
}

IG_DEV bool run_bfs(const BatchTask& T, const Team& tm, unsigned long long (*s_acc)[kWave],
                    BlockQueue<kBatchQueue>& s_next, BlockSum& s_mf)
{
  const int V = T.nodes;
  const int lane = lane_id();
  const size_t Vs = static_cast<size_t>(V);
  unsigned long long* seen = static_cast<unsigned long long*>(T.scratch);
  unsigned long long* fr[2] = {seen + Vs, seen + 2 * Vs};  // frontier masks by level parity
  unsigned long long* nxt = seen + 3 * Vs;                 // next-level masks
  int* queue0 = reinterpret_cast<int*>(seen + 4 * Vs);
  unsigned* qn = tm.gs->qn;
  unsigned long long* mf = tm.gs->mf;
  const unsigned long long all = T.nsrc >= 64 ? ~0ull : ((1ull << T.nsrc) - 1ull);
  const Chunks ch = team_chunks(tm, V);
  for (int c = ch.first; c < ch.count; c += ch.step) {
    const int v = c * kWave + lane;
    if (v < V) {
      st_relaxed(&seen[v], 0ull);
      st_relaxed(&fr[0][v], 0ull);
      st_relaxed(&fr[1][v], 0ull);
      st_relaxed(&nxt[v], 0ull);
    }
  }
  int nitems = 0;
  if (!build_items(T, tm, &nitems)) return false;
  if (tm.rank == 0 && threadIdx.x < kWave) {  // one wave queues the distinct sources
    const bool has = lane < T.nsrc;
    const int i = lane;
    const int s = has ? T.src[i] : 0;
    unsigned long long old = 0ull;
    if (has) {
      __hip_atomic_fetch_or(&seen[s], 1ull << i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      old = __hip_atomic_fetch_or(&fr[0][s], 1ull << i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      st_relaxed(&T.out[static_cast<size_t>(i) * V + s], 0);
    }
    // a source listed twice is queued by the lane that set its first bit
    const bool first = has && old == 0ull;
    wave_append(first, s, queue0, &qn[0]);
    const unsigned long long d = wave_sum(static_cast<unsigned long long>(first ? T.nindex[s + 1] - T.nindex[s] : 0));
    if (lane == 0) atomic_add_relaxed(&mf[0], d);
  }
  if (!team_sync(tm)) return false;
  int ncur = static_cast<int>(ld_relaxed(&qn[0]));
  unsigned long long mcur = ld_relaxed(&mf[0]);
  // (member 0 may go ahead from here: all have read the counters)
  if (tm.size > 1 && !team_sync(tm)) return false;
  for (int lvl = 1;; lvl++) {
    // narrow levels are member 0's, at workgroup barriers, until one is wider; the
    // others wait for it (a chain of 4096 cliques of 12, on the 128 members that its
    // entries give it: 75 ms a BFS, now 29)
    const bool solo = tm.size > 1 && mcur <= kNarrow;
    Team w = tm;
    w.size = solo ? 1 : tm.size;  // (member 0 keeps its rank)
    int nnext = 0;
    unsigned long long mnext = 0ull;
    if (solo && tm.rank != 0) {
      if (!team_sync(tm)) return false;
      lvl = static_cast<int>(ld_relaxed(&tm.gs->flag[0]));
      nnext = static_cast<int>(ld_relaxed(&qn[lvl & 3]));
      mnext = ld_relaxed(&mf[lvl & 3]);
    } else if (!bfs_level(T, w, lvl, nitems, all, ncur, mcur, &nnext, &mnext, s_acc, s_next, s_mf)) {
      return false;
    } else if (solo && (nnext == 0 || mnext > kNarrow)) {
      if (threadIdx.x == 0) st_relaxed(&tm.gs->flag[0], static_cast<unsigned>(lvl));
      if (!team_sync(tm)) return false;
    }
    if (nnext == 0) break;
    ncur = nnext;
    mcur = mnext;
  }
  for (int c = ch.first; c < ch.count; c += ch.step) {
    const int v = c * kWave + lane;
    write_rows(T, v < V ? all & ~ld_relaxed(&seen[v]) : 0ull, v, INT_MAX);
  }
  return true;
}

// ---- multi-source SSSP -------------------------------------------------------
// The distances live vertex-major, row[v * G + i] for source i (G = nsrc rounded up
// to a power of two), so an entry's are runs of consecutive words; they are turned into
// the output's source-major slab at the end.  A queued vertex has its active sources,
// those whose distance fell in the round before, in a mask.  relax_lists has how a wave
// takes its vertices' lists.  With a lane per entry that walked its sources over
// source-major rows, every distance was a line of its own: 1024 queries of 16 sources on
// random graphs of 2^13 vertices and degree 32 255 ms, now 62; R-MAT 14 97 -> 37; 24 uneven
// graphs, all algorithms, 61 -> 5.9.  What is bound by latency instead gains little, or
// loses: gangs of one 0.8 to 1.6 times as fast, 1024 trees of 2^13 vertices with 32 sources,
// where every distance falls once, 8.3 -> 11.7 ms.  (Deferring distances above a
// threshold that grows by twice the mean weight over the degree a round saved relaxations
// but no time.)  Split lists are split into short items, each entry being nsrc pairs.
// Sources are taken T.rows at a time, all of them where the rows fit the memory.

// The n-th (from 0) set bit of m.
IG_DEV int nth_bit(unsigned m, int n)
{
  int pos = 0;
#pragma unroll
  for (int half = 16; half > 0; half >>= 1) {
    const int low = __popc(m & ((1u << half) - 1u));
    if (n >= low) {
      n -= low;
      m >>= half;
      pos += half;
    }
  }
  return pos;
}

struct SsspRows {
  int* row;        // [V << shift]
  unsigned* mask;  // [V] sources active in the next round
  int shift;
  bool direct;  // narrow round: appends go straight to the queue
  int* qnext;
  unsigned* ncount;
};

constexpr unsigned long long kTwoInf = 0x7fffffff7fffffffull;  // two entries of INT_MAX

IG_DEV int* row_of(const SsspRows& R, int v, int i) { return &R.row[(static_cast<size_t>(v) << R.shift) + i]; }

// A wave's block of 64 list entries: neighbour, weight, owner and the owner's active
// sources; and the sources for which the neighbour's distance fell.
struct SsspBlock {
  int4 entry[kWave];
  unsigned gain[kWave];
};

// Wave-collective: relaxes each lane's list [beg, beg + len) of vertex v for the
// sources in m, in blocks of 64 entries: an entry per lane is looked up, the block's
// (entry, source) pairs are relaxed, and each entry's improvements are added to its
// neighbour's mask for the next round, with one atomic and, where the mask was
// empty, one append to the queue.  (Both with every step of the pairs: a gang of one on
// a star of 2^18 leaves 19.6 ms for 16 sources, by the block 8.4.)
//
// The pairs of a block are taken in one of three ways, by how many sources are active:
//   * at most kLaneFly per entry: by the entry's lane, all loads in flight together (16
//     sources on a path: 4.7 us a round by pairs, 3.5);
//   * half of all: 64 >> shift entries a step, a lane for each source, active or not (what
//     has not fallen since it was last relaxed improves nothing);
//   * else exactly the active pairs, one per lane, which finds its entry and source with
//     7 permutes through LDS (left to the entries' lanes, R-MAT 14 as above took 53 ms).
// More steps in flight than this spill registers: 24 graphs 5.9 -> 6.2 ms.
IG_DEV void relax_lists(const BatchTask& T, const SsspRows& R, int v, int beg, int len, unsigned m, SsspBlock& B,
                        BlockQueue<kBatchQueue>& s_next)
{
  const int lane = lane_id();
  const int entries = m != 0u ? len : 0;
  const int incl = wave_inclusive_scan(entries);
  const int count = wave_bcast(incl, kWave - 1);
  for (int base = 0; base < count; base += kWave) {
    const int k = base + lane;
    const int o = min(wave_owner(incl, k), kWave - 1);
    const int ov = wave_shfl(v, o);
    const unsigned om = static_cast<unsigned>(wave_shfl(static_cast<int>(m), o));
    const int e = wave_shfl(beg - (incl - entries), o) + k;
    int4 mine = make_int4(0, 0, ov, 0);
    if (k < count) {
      mine.x = T.nlist[e];
      mine.y = T.eweight[e];
      mine.w = static_cast<int>(om);
    }
    const int left = min(kWave, count - base);
    const int pop = __popc(static_cast<unsigned>(mine.w));
    unsigned gain = 0u;
    if (__ballot(pop > kLaneFly) == 0ull) {
      unsigned bits = static_cast<unsigned>(mine.w);
      int i[kLaneFly], d[kLaneFly], old[kLaneFly];
#pragma unroll
      for (int q = 0; q < kLaneFly; q++) {
        i[q] = bits != 0u ? __ffs(static_cast<int>(bits)) - 1 : 0;
        d[q] = bits != 0u ? ld_relaxed(row_of(R, ov, i[q])) : 0;
        old[q] = bits != 0u ? ld_relaxed(row_of(R, mine.x, i[q])) : INT_MIN;
        bits &= bits - 1u;
      }
#pragma unroll
      for (int q = 0; q < kLaneFly; q++) {
        const int nd = d[q] + mine.y;
        if (nd < old[q]) {
          atomic_min_relaxed(row_of(R, mine.x, i[q]), nd);
          gain |= 1u << i[q];
        }
      }
    } else {
      B.entry[lane] = mine;
      B.gain[lane] = 0u;
      const int pair_incl = wave_inclusive_scan(pop);
      const int pairs = wave_bcast(pair_incl, kWave - 1);
      wave_lds_sync();
      if ((left << R.shift) <= 2 * pairs) {
        const int per = kWave >> R.shift;  // entries a step
        const int src = lane & ((1 << R.shift) - 1);
        const unsigned group = R.shift == 5 ? ~0u : (1u << (1 << R.shift)) - 1u;
        for (int j = 0; j < left; j += kGroupFly * per) {
          int at[kGroupFly], d[kGroupFly], old[kGroupFly];
          int2 to[kGroupFly];  // neighbour, weight
#pragma unroll
          for (int q = 0; q < kGroupFly; q++) {
            at[q] = j + q * per + (lane >> R.shift);
            const int4 entry = B.entry[min(at[q], kWave - 1)];
            to[q] = make_int2(entry.x, entry.y);
            d[q] = at[q] < left ? ld_relaxed(row_of(R, entry.z, src)) : INT_MAX;
            old[q] = at[q] < left ? ld_relaxed(row_of(R, entry.x, src)) : INT_MIN;
          }
#pragma unroll
          for (int q = 0; q < kGroupFly; q++) {
            const int nd = d[q] + to[q].y;
            const bool on = d[q] != INT_MAX && nd < old[q];
            const unsigned long long all = __ballot(on);
            if (on) atomic_min_relaxed(row_of(R, to[q].x, src), nd);
            if (src == 0 && at[q] < left) B.gain[at[q]] = static_cast<unsigned>(all >> lane) & group;
          }
        }
      } else {
        for (int p0 = 0; p0 < pairs; p0 += kWave) {
          const int p = p0 + lane;
          const int at = min(wave_owner(pair_incl, p), kWave - 1);
          const int rank = p - wave_shfl(pair_incl - pop, at);
          const int4 entry = B.entry[at];
          const int i = nth_bit(static_cast<unsigned>(entry.w), rank) & 31;  // (any, past the pairs)
          const int d = p < pairs ? ld_relaxed(row_of(R, entry.z, i)) : 0;
          const int old = p < pairs ? ld_relaxed(row_of(R, entry.x, i)) : INT_MIN;
          if (d + entry.y < old) {
            atomic_min_relaxed(row_of(R, entry.x, i), d + entry.y);
            atomicOr(&B.gain[at], 1u << i);
          }
        }
      }
      wave_lds_sync();
      gain = B.gain[lane];
    }
    // (whether or not this wave's minimum is the one that lowered a distance: one of
    // this round's is)
    const bool first = gain != 0u && __hip_atomic_fetch_or(&R.mask[mine.x], gain, __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_AGENT) == 0u;
    if (R.direct) wave_append(first, mine.x, R.qnext, R.ncount);
    else bq_append(s_next, first, mine.x, R.qnext, R.ncount);
  }
}

// Gang-collective over the members of w: round r over its queue of ncur vertices; *count gets
// the next one's.
IG_DEV bool sssp_round(const BatchTask& T, const Team& w, SsspRows& R, unsigned* base, int r, int nitems, int ncur,
                       int* count, SsspBlock& B, BlockQueue<kBatchQueue>& s_next)
{
  const int lane = lane_id();
  const size_t Vs = static_cast<size_t>(T.nodes);
  unsigned* act[3] = {base, base + Vs, base + 2 * Vs};  // masks of active sources by round mod 3
  int* queue[2] = {reinterpret_cast<int*>(base + 3 * Vs), reinterpret_cast<int*>(base + 4 * Vs)};
  unsigned* qn = w.gs->qn;
  const Chunks ch = team_chunks(w, T.nodes);
  unsigned* cur = act[r % 3];
  const int* qcur = queue[r & 1];
  R.mask = act[(r + 1) % 3];
  R.qnext = queue[(r + 1) & 1];
  R.ncount = &qn[(r + 1) & 3];
  if (w.rank == 0 && threadIdx.x == 0) st_relaxed(&qn[(r + 2) & 3], 0u);
  R.direct = ncur <= kWave;  // (as a BFS's narrow levels)
  if (!R.direct) bq_reset(s_next);
  // few queued vertices: fewer per wave
  int per = kWave;
  while (per > 4 && ncur <= per / 2 * ch.step) per /= 2;
  // the queue, then the items of split lists, a lane each
  for (int c = ch.first, i0 = ch.first;;) {
    int v = 0, beg = 0, len = 0;
    unsigned m = 0u;
    if (c * per < ncur) {
      const int k = c * per + lane;
      if (lane < per && k < ncur) {
        v = ld_relaxed(&qcur[k]);
        m = ld_relaxed(&cur[v]);
        beg = T.nindex[v];
        len = T.nindex[v + 1] - beg;
        if (len >= T.item) len = 0;
        if (len > 0) st_relaxed(&cur[v], 0u);  // (no one else reads it)
      }
      c += ch.step;
    } else if (i0 < nitems) {
      const int i = i0 + lane * ch.step;
      if (i < nitems) {
        v = ld_relaxed(&T.items[i].x);
        beg = ld_relaxed(&T.items[i].y);
        m = ld_relaxed(&cur[v]);
        len = min(T.item, T.nindex[v + 1] - beg);
        if (beg == T.nindex[v]) st_relaxed(&act[(r + 2) % 3][v], 0u);  // the last round's
      }
      i0 += kWave * ch.step;
    } else {
      break;
    }
    relax_lists(T, R, v, beg, len, m, B, s_next);
  }
  if (!R.direct) bq_flush<false>(s_next, R.qnext, R.ncount);
  if (!team_sync(w)) return false;
  *count = static_cast<int>(ld_relaxed(R.ncount));
  return true;
}

// One pass: the distances from the sources [s0, s0 + n).
IG_DEV bool sssp_pass(const BatchTask& T, const Team& tm, int s0, int n, int* nitems, SsspBlock& B,
                      BlockQueue<kBatchQueue>& s_next)
{
  const int V = T.nodes;
  const int lane = lane_id();
  const size_t Vs = static_cast<size_t>(V);
  SsspRows R;
  R.shift = sssp_row_shift(T.rows);
  // (one source a pass: the distances are its slab row)
  R.row = T.rows == 1 ? T.out + s0 * Vs : static_cast<int*>(T.scratch);
  unsigned* base = static_cast<unsigned*>(T.scratch) + (T.rows == 1 ? 0 : Vs << R.shift);
  unsigned* qn = tm.gs->qn;
  const Chunks ch = team_chunks(tm, V);
  for (int c = ch.first; c < ch.count; c += ch.step) {
    const int v = c * kWave + lane;
    if (v < V) {
      st_relaxed(&base[v], 0u);
      st_relaxed(&base[Vs + v], 0u);
      st_relaxed(&base[2 * Vs + v], 0u);
    }
    if (T.rows == 1) {
      if (v < V) st_relaxed(&R.row[v], INT_MAX);
    } else {
      const size_t end = min(Vs, static_cast<size_t>(c + 1) * kWave) << R.shift >> 1;
      for (size_t k = (static_cast<size_t>(c) * kWave << R.shift >> 1) + lane; k < end; k += kWave)
        st_relaxed(reinterpret_cast<unsigned long long*>(R.row) + k, kTwoInf);
    }
  }
  if (tm.rank == 0 && threadIdx.x < 4) st_relaxed(&qn[threadIdx.x], 0u);
  if (s0 == 0) {
    if (!build_items(T, tm, nitems)) return false;  // (ends with a team barrier)
  } else if (!team_sync(tm)) {
    return false;
  }
  if (tm.rank == 0 && threadIdx.x < kWave) {
    const bool has = lane < n;
    const int s = has ? T.src[s0 + lane] : 0;
    unsigned old = 1u;
    if (has) {
      st_relaxed(&R.row[(static_cast<size_t>(s) << R.shift) + lane], 0);
      old = __hip_atomic_fetch_or(&base[s], 1u << lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    wave_append(old == 0u, s, reinterpret_cast<int*>(base + 3 * Vs), &qn[0]);
  }
  if (!team_sync(tm)) return false;
  int ncur = static_cast<int>(ld_relaxed(&qn[0]));
  bool solo = false;
  for (int r = 0;; r++) {
    // narrow rounds are member 0's, as a BFS's narrow levels (unless lists are split); here all
    // meet before it goes ahead, having read the count
    if (!solo && tm.size > 1 && *nitems == 0 && ncur <= kNarrowQueue) {
      solo = true;
      if (!team_sync(tm)) return false;
    }
    int count = 0;
    if (solo && tm.rank != 0) {
      if (!team_sync(tm)) return false;
      solo = false;
      r = static_cast<int>(ld_relaxed(&tm.gs->flag[0]));
      count = static_cast<int>(ld_relaxed(&qn[(r + 1) & 3]));
    } else {
      Team w = tm;
      w.size = solo ? 1 : tm.size;
      if (!sssp_round(T, w, R, base, r, *nitems, ncur, &count, B, s_next)) return false;
      if (solo && (count == 0 || count > 4 * kNarrowQueue)) {
        if (threadIdx.x == 0) st_relaxed(&tm.gs->flag[0], static_cast<unsigned>(r));
        if (!team_sync(tm)) return false;
        solo = false;
      }
    }
    if (count == 0) break;
    ncur = count;
  }
  if (T.rows == 1) return true;
  for (int c = ch.first; c < ch.count; c += ch.step) {
    const int v = c * kWave + lane;
    if (v >= V) continue;
    for (int i = 0; i < n; i += 2) {
      const unsigned long long two = ld_relaxed(reinterpret_cast<unsigned long long*>(row_of(R, v, i)));
      T.out[(s0 + i) * Vs + v] = static_cast<int>(two);
      if (i + 1 < n) T.out[(s0 + i + 1) * Vs + v] = static_cast<int>(two >> 32);
    }
  }
  return true;
}

IG_DEV bool run_sssp(const BatchTask& T, const Team& tm, SsspBlock* s_block, BlockQueue<kBatchQueue>& s_next)
{
  int nitems = 0;
  for (int s0 = 0; s0 < T.nsrc; s0 += T.rows)
    if (!sssp_pass(T, tm, s0, min(T.rows, T.nsrc - s0), &nitems, s_block[threadIdx.x / kWave], s_next)) return false;
  return true;
}

// ---- CC ------------------------------------------------------------------------
// Root of x without find_root's store.  The final flatten writes roots into the
// same array the finds walk: a store of what was the root when the walk read it
// could land over the flattened entry, so that pass stores final roots only.
IG_DEV int root_of(const int* parent, int x)
{
  int p;
  while ((p = ld_relaxed(&parent[x])) != x) x = p;
  return x;
}

// Workgroup-collective: the most frequent root among kCcSamples vertices
// spread over the id range (ties to the smaller root).  Every gang member
// reads the same compressed parents, so all choose the same root.
IG_DEV int giant_root(const BatchTask& T, int* parent, unsigned long long (*s_acc)[kWave])
{
  int* s_root = reinterpret_cast<int*>(&s_acc[0][0]);  // kCcSamples ints of the task scratch LDS
  const int V = T.nodes;
  for (int i = threadIdx.x; i < kCcSamples; i += blockDim.x)
    s_root[i] = find_root<kCcDepth>(parent, static_cast<int>((static_cast<unsigned long long>(i) * 2654435761ull) %
                                                   static_cast<unsigned>(V)));
  __syncthreads();
  unsigned long long key = 0;  // (count << 32) | ~root: the largest wins
  for (int i = threadIdx.x; i < kCcSamples; i += blockDim.x) {
    unsigned c = 0;
    for (int j = 0; j < kCcSamples; j++) c += s_root[j] == s_root[i] ? 1u : 0u;
    const unsigned long long k = (static_cast<unsigned long long>(c) << 32) | (~static_cast<unsigned>(s_root[i]));
    key = k > key ? k : key;
  }
  __syncthreads();
  key = wave_max(key);
  if (lane_id() == 0) s_acc[threadIdx.x / kWave][0] = key;
  __syncthreads();
  unsigned long long best = 0;
  for (int w = 0; w < kBatchWaves; w++) best = s_acc[w][0] > best ? s_acc[w][0] : best;
  __syncthreads();
  return static_cast<int>(~static_cast<unsigned>(best & 0xffffffffull));
}

// CC as the single-query kernel: union-find hooking the larger root under
// the smaller (labels = component minima).  Graphs with an average degree of
// at least 8 (and kCcAfforestMin vertices) take the Afforest order - link
// each vertex with its first kCcSample neighbours, compress, choose the giant
// root, and let only vertices outside its tree link their lists (all
// entries); the others link every undirected edge once, from its larger
// endpoint.
IG_DEV bool run_cc(const BatchTask& T, const Team& tm, unsigned long long (*s_acc)[kWave])
{
  const int V = T.nodes;
  const int lane = lane_id();
  int* parent = T.out;
  const bool aff = static_cast<long long>(T.edges) >= 8LL * V && V >= kCcAfforestMin;
  const Chunks ch = team_chunks(tm, V);
  for (int c = ch.first; c < ch.count; c += ch.step) {
    const int v = c * kWave + lane;
    if (v < V) {
      int p = v;
      if (aff && T.nindex[v] < T.nindex[v + 1]) p = min(v, T.nlist[T.nindex[v]]);
      st_relaxed(&parent[v], p);
    }
  }
  int nitems = 0;
  if (!build_items(T, tm, &nitems)) return false;  // (ends with a team barrier)
  int giant = -1;
  if (aff) {
    for (int c = ch.first; c < ch.count; c += ch.step) {
      const int v = c * kWave + lane;
      if (v < V) {
        const int b = T.nindex[v], e = min(T.nindex[v + 1], b + kCcSample);
        for (int k = b; k < e; k++) link<kCcDepth>(parent, v, T.nlist[k]);
      }
    }
    if (!team_sync(tm)) return false;
    for (int c = ch.first; c < ch.count; c += ch.step) {
      const int v = c * kWave + lane;
      if (v < V) st_relaxed(&parent[v], find_root<kCcDepth>(parent, v));
    }
    if (!team_sync(tm)) return false;
    giant = giant_root(T, parent, s_acc);
    // Nobody links before all have chosen: a member that sampled parents another
    // had begun to hook could choose another root, and of an edge between the two
    // roots' trees each end would be skipped, by the member that chose its tree.
    if (!team_sync(tm)) return false;
  }
  for (int c = ch.first; c < ch.count; c += ch.step) {
    const int v = c * kWave + lane;
    bool todo = v < V;
    if (aff && todo) todo = T.nindex[v + 1] - T.nindex[v] > kCcSample && find_root<kCcDepth>(parent, v) != giant;
    wave_entries_of(v, todo, T.nindex, [&](int o, int e, bool valid) {
      if (!valid) return;
      const int ov = c * kWave + o;
      const int u = T.nlist[e];
      if (aff || u < ov) link<kCcDepth>(parent, ov, u);
    });
  }
  for_items(T, tm, nitems, [&](int v, int eb, int ee, int) {
    if (aff && find_root<kCcDepth>(parent, v) == giant) return;
    for (int e = eb + lane; e < ee; e += kWave) {
      const int u = T.nlist[e];
      if (aff || u < v) link<kCcDepth>(parent, v, u);
    }
  });
  if (!team_sync(tm)) return false;
  for (int c = ch.first; c < ch.count; c += ch.step) {
    const int v = c * kWave + lane;
    if (v < V) st_relaxed(&parent[v], root_of(parent, v));
  }
  return true;
}

// ---- MIS -------------------------------------------------------------------------
struct MisView {
  const int* nlist;
  int* status;
  unsigned flip;
};

// Rounds of decisions in place, as the single-query kernel's: a lane looks at the
// first entries of a list, eight lanes (a wave from kMisWaveList entries on) finish
// what they leave open, and a vertex that joins excludes its smaller neighbours.  A
// heavy vertex's items gather flags (1: a larger neighbour not excluded, 2: one
// included), by which its own chunk decides it in the next round; the flags of
// even and odd rounds are apart.  One barrier a round.  (Rounds of two phases that
// each read all entries of the undecided vertices: 12.6 ms for 100 graphs, now 2.6.)
IG_DEV bool run_mis(const BatchTask& T, const Team& tm)
{
  const int V = T.nodes;
  const int lane = lane_id();
  const MisView a{T.nlist, T.out, 0u};
  unsigned* flags[2] = {static_cast<unsigned*>(T.scratch), static_cast<unsigned*>(T.scratch) + V};
  const Chunks ch = team_chunks(tm, V);
  for (int c = ch.first; c < ch.count; c += ch.step) {
    const int v = c * kWave + lane;
    if (v < V) {
      st_relaxed(&a.status[v], kUndecided);
      st_relaxed(&flags[0][v], 0u);
      st_relaxed(&flags[1][v], 0u);
    }
  }
  int nitems = 0;
  if (!build_items(T, tm, &nitems)) return false;
  for (int r = 0;; r++) {
    unsigned* flag = &tm.gs->flag[r % 3];
    if (tm.rank == 0 && threadIdx.x == 0) st_relaxed(&tm.gs->flag[(r + 1) % 3], 0u);
    unsigned* seen = flags[(r + 1) & 1];  // the last round's flags
    bool still = false;
    for (int c = ch.first; c < ch.count; c += ch.step) {
      const int v = c * kWave + lane;
      const bool und = v < V && ld_relaxed(&a.status[v]) == kUndecided;
      if (__ballot(und) == 0ull) continue;
      const int beg = und ? T.nindex[v] : 0;
      const int end = und ? T.nindex[v + 1] : 0;
      bool rest = false;
      if (und) {
        int st = kUndecided;
        if (!heavy(end - beg)) {
          st = decide_lane(a, v, beg, end);
          rest = st < 0;
        } else if (r > 0) {
          const unsigned f = ld_relaxed(&seen[v]);
          st_relaxed(&seen[v], 0u);
          st = (f & 2u) != 0u ? kExcluded : ((f & 1u) != 0u ? kUndecided : kIncluded);
        }
        if (st == kIncluded || st == kExcluded) st_relaxed(&a.status[v], st);
        if (st == kIncluded && !heavy(end - beg)) exclude_neighbours_lane(a, v, beg, end);
        still |= st == kUndecided;
      }
      constexpr int kPer = kWave >> kMisGroupShift;
      const bool grouped = rest && end - beg < kMisWaveList;
      const unsigned long long m = __ballot(grouped);
      const int rows = __popcll(m), rank = lanes_below(m);
      const int of = __builtin_amdgcn_ds_permute((grouped ? rank : lane - rank + rows) << 2, lane);
      for (int r0 = 0; r0 < rows; r0 += kPer) {
        const int row = r0 + (lane >> kMisGroupShift);
        const int o = wave_shfl(of, min(row, kWave - 1));
        const int gv = wave_shfl(v, o), gb = wave_shfl(beg, o), ge = wave_shfl(end, o);
        still |= decide_group(a, gv, gb, gb + kMisLaneUnroll, row < rows ? ge : gb, kMisGroupShift) == kUndecided;
      }
      for (unsigned long long w = __ballot(rest && !grouped); w != 0ull; w &= w - 1ull) {
        const int o = __ffsll(static_cast<long long>(w)) - 1;
        const int wb = wave_bcast(beg, o);
        still |= decide_group(a, wave_bcast(v, o), wb, wb + kMisLaneUnroll, wave_bcast(end, o), 6) == kUndecided;
      }
    }
    set_flag(flag, still);
    for_items(T, tm, nitems, [&](int v, int eb, int ee, int) {
      if (ld_relaxed(&a.status[v]) != kUndecided) return;
      const unsigned long long kv = mis_key(v, a.flip);
      unsigned f = 0u;
      for (int e = eb + lane; e < ee; e += kWave) {
        const int u = T.nlist[e];
        if (u == v || mis_key(u, a.flip) < kv) continue;  // smaller keys cannot decide v
        const int su = ld_relaxed(&a.status[u]);
        f |= su == kIncluded ? 3u : (su == kUndecided ? 1u : 0u);
      }
      f = (__ballot((f & 1u) != 0u) != 0ull ? 1u : 0u) | (__ballot((f & 2u) != 0u) != 0ull ? 2u : 0u);
      if (lane == 0 && f != 0u)
        __hip_atomic_fetch_or(&flags[r & 1][v], f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    });
    if (!team_sync(tm)) return false;
    if (ld_relaxed(flag) == 0u) break;
  }
  return true;
}

// ---- PageRank ----------------------------------------------------------------------
// Bound by the latency of the gathers.  Four masked loads per lane in flight and
// groups of lanes for lists of 8 to 63 entries, as in the single-query kernel
// (one lane or a wave per list, a load at a time: 52 -> 36 ms for 100 graphs).
IG_DEV bool run_pr(const BatchTask& T, const Team& tm, double* s_red)
{
  const int V = T.nodes;
  const int lane = lane_id();
  const int wid = threadIdx.x / kWave;
  const size_t Vs = static_cast<size_t>(V);
  float* scores = reinterpret_cast<float*>(T.out);
  double* slots = static_cast<double*>(T.scratch);  // [2][kMaxGang] FP64 partials
  float* contrib[2] = {reinterpret_cast<float*>(slots + 2 * kMaxGang),
                       reinterpret_cast<float*>(slots + 2 * kMaxGang) + Vs};
  float2* hpart = reinterpret_cast<float2*>(contrib[1] + Vs);  // per item (sum, error)
  const float inv_n = 1.0f / static_cast<float>(V);
  const float base = (1.0f - kDamp) / static_cast<float>(V);
  const Chunks ch = team_chunks(tm, V);
  for (int c = ch.first; c < ch.count; c += ch.step) {
    const int v = c * kWave + lane;
    if (v >= V) continue;
    st_relaxed(&scores[v], inv_n);
    st_relaxed(&contrib[0][v], inv_n / static_cast<float>(T.nindex[v + 1] - T.nindex[v]));
  }
  int nitems = 0;
  if (!build_items(T, tm, &nitems)) return false;
  // a heavy vertex's score is written at init by its chunk's wave and later by
  // the wave of its first item, possibly on another XCD: device-scope stores
  // keep the two L2s from writing back stale bytes
  auto finish = [&](float* cout, int x, int xdeg, float total) {
    const float old = ld_relaxed(&scores[x]);
    const float s = base + kDamp * total;
    st_relaxed(&scores[x], s);
    st_relaxed(&cout[x], s / static_cast<float>(xdeg));
    return fabs(static_cast<double>(s) - static_cast<double>(old));
  };
  int it = 0;
  for (;;) {
    it++;
    const float* cin = contrib[(it - 1) & 1];
    float* cout = contrib[it & 1];
    auto contribution = [cin](int u) { return ld_relaxed(&cin[u]); };
    double d = 0.0;
    for (int c = ch.first; c < ch.count; c += ch.step) {
      const int v = c * kWave + lane;
      const int beg = v < V ? T.nindex[v] : 0;
      const int deg = v < V ? T.nindex[v + 1] - beg : 0;
      const float sum = short_sums(contribution, T.nlist, beg, beg + deg, false);
      if (v < V && deg < kPrWaveDeg) d += finish(cout, v, deg, sum);
      for (unsigned long long m = __ballot(deg >= kPrWaveDeg && !heavy(deg)); m != 0ull; m &= m - 1ull) {
        const int o = __ffsll(static_cast<long long>(m)) - 1;
        const int x = c * kWave + o;
        const int xb = wave_bcast(beg, o), xd = wave_bcast(deg, o);
        CSum acc;
        gather<kWave>(acc, contribution, T.nlist, xb, xb + xd, lane);
        acc = wave_merge(acc);
        if (lane == 0) d += finish(cout, x, xd, acc.value());
      }
    }
    if (nitems > 0) {
      for_items(T, tm, nitems, [&](int, int eb, int ee, int i) {
        CSum acc;
        gather<kWave>(acc, contribution, T.nlist, eb, ee, lane);
        acc = wave_merge(acc);
        if (lane == 0) {
          st_relaxed(&hpart[i].x, acc.s);
          st_relaxed(&hpart[i].y, acc.c);
        }
      });
      if (!team_sync(tm)) return false;
      // one wave per heavy vertex (at its first item) combines its items in order
      for_items(T, tm, nitems, [&](int v, int eb, int, int i) {
        if (eb != T.nindex[v]) return;
        const int deg = T.nindex[v + 1] - eb;
        const int n = (deg + kItem - 1) / kItem;
        CSum acc;
        for (int j = lane; j < n; j += kWave) acc.merge(ld_relaxed(&hpart[i + j].x), ld_relaxed(&hpart[i + j].y));
        acc = wave_merge(acc);
        if (lane == 0) d += finish(cout, v, deg, acc.value());
      });
    }
    // the member's FP64 partial (fixed order: wave tree, then waves in order)
    d = wave_sum(d);
    if (lane == 0) s_red[wid] = d;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
      for (int w = 0; w < kBatchWaves; w++) t += s_red[w];
      st_relaxed(&slots[(it & 1) * kMaxGang + tm.rank], t);
    }
    if (!team_sync(tm)) return false;
    double total = 0.0;
    for (int r = 0; r < tm.size; r++) total += ld_relaxed(&slots[(it & 1) * kMaxGang + r]);
    if (!(total > static_cast<double>(0.0001f) && it < 100)) break;
  }
  if (tm.rank == 0 && threadIdx.x == 0) st_relaxed(&T.out[V], it);
  return true;
}

__global__ __launch_bounds__(kBatchBlock) __attribute__((amdgpu_waves_per_eu(8, 8))) IG_SGPR_CAP void batch_kernel(const BatchTask* __restrict__ tasks, int ntasks,
                                                            GangState* gangs, BatchControl* ctl, long long budget,
                                                            long long residency_ticks)
{
  __shared__ int s_task, s_rank;
  __shared__ union {
    unsigned long long acc[kBatchWaves][kWave];  // BFS, CC
    SsspBlock block[kBatchWaves];                // SSSP
  } s_wave;
  __shared__ double s_red[kBatchWaves];
  __shared__ BlockQueue<kBatchQueue> s_next;
  __shared__ BlockSum s_mf;
  if (!residency_barrier(&ctl->bar, residency_ticks)) return;
  const long long deadline = now_ticks() + budget;
  for (;;) {
    if (threadIdx.x == 0) {
      int t = static_cast<int>(ld_relaxed(&ctl->head));
      int rank = -1;
      while (t < ntasks) {
        const unsigned r = atomic_add_relaxed(&gangs[t].joined, 1u);
        if (r < static_cast<unsigned>(min(tasks[t].gang, static_cast<int>(gridDim.x)))) {
          rank = static_cast<int>(r);
          break;
        }
        atomic_max_relaxed(&ctl->head, static_cast<unsigned>(t + 1));
        t++;
      }
      s_task = t;
      s_rank = rank;
    }
    __syncthreads();
    const int t = s_task;
    const int rank = s_rank;
    __syncthreads();
    if (t >= ntasks) break;
    const BatchTask& T = tasks[t];
    // a relaunch after a failed residency check may run a smaller grid
    const Team tm{rank, min(T.gang, static_cast<int>(gridDim.x)), &gangs[t], &ctl->bar, deadline};
    if (!team_sync(tm)) break;  // the gang assembles
    bool ok = true;
    if (T.alg == INDIGO_QUERY_BFS) ok = run_bfs(T, tm, s_wave.acc, s_next, s_mf);
    else if (T.alg == INDIGO_QUERY_SSSP) ok = run_sssp(T, tm, s_wave.block, s_next);
    else if (T.alg == INDIGO_QUERY_CC) ok = run_cc(T, tm, s_wave.acc);
    else if (T.alg == INDIGO_QUERY_PR) ok = run_pr(T, tm, s_red);
    else ok = run_mis(T, tm);
    if (!ok) break;
  }
}

// Sources that one pass of an SSSP takes, at most `most` (a power of two).
int pass_rows(const indigo_query& Q, int most)
{
  return Q.alg == INDIGO_QUERY_SSSP ? std::min(1 << sssp_row_shift(Q.nsrc), most) : 1;
}

// Entries per item: lists that long tie a wave up.  An entry of a multi-source SSSP
// is a pair per source, so its items hold about kItem pairs.
int item_entries(int alg, int rows)
{
  return alg == INDIGO_QUERY_SSSP ? std::max(kWave, kItem >> sssp_row_shift(rows)) : kItem;
}

size_t items_cap(int edges, int item) { return 2 * (static_cast<size_t>(edges) / item) + 2; }

// Per-task scratch: the algorithm's arrays (alg_bytes), then the heavy items.
size_t alg_bytes(int alg, int nodes, int edges, int rows)
{
  const size_t v = static_cast<size_t>(nodes);
  size_t b = 0;
  if (alg == INDIGO_QUERY_BFS) b = 4 * v * 8 + 2 * v * 4;             // seen, 2 frontiers, next; 2 queues
  else if (alg == INDIGO_QUERY_SSSP) b = 5 * v * 4 + (rows == 1 ? 0 : v * 4 * rows);  // 3 masks, 2 queues; rows
  else if (alg == INDIGO_QUERY_MIS) b = 2 * v * 4;                   // heavy-vertex flags
  else if (alg == INDIGO_QUERY_PR) b = 2 * kMaxGang * 8 + 2 * v * 4 + items_cap(edges, kItem) * 8;  // slots, contrib, partials
  return Carver::round(b);
}

size_t scratch_bytes(int alg, int nodes, int edges, int rows)
{
  return alg_bytes(alg, nodes, edges, rows) + Carver::round(items_cap(edges, item_entries(alg, rows)) * sizeof(int2));
}

// Workspace of a batch whose SSSPs take at most `most` sources a pass.
size_t workspace_bytes(const indigo_graph_ref* graphs, const indigo_query* queries, int nqueries, int most)
{
  const size_t n = static_cast<size_t>(nqueries);
  size_t bytes = Carver::round(sizeof(BatchControl)) + Carver::round(n * sizeof(GangState)) +
                 Carver::round(n * sizeof(BatchTask)) + 4096;
  for (int q = 0; q < nqueries; q++) {
    const indigo_graph_ref& G = graphs[queries[q].graph];
    bytes += scratch_bytes(queries[q].alg, G.nodes, G.edges, pass_rows(queries[q], most));
  }
  return bytes;
}

}  // namespace

// Largest gang of an algorithm: how much work one of its barriers separates.  An
// SSSP of many sources goes on gaining past 64 members, but only workgroups that
// have nothing else to do take it there (widen_gangs).
static int gang_cap(int alg, int nodes, int edges, bool widen)
{
  if (alg == INDIGO_QUERY_SSSP) return widen ? kMaxGang : 64;
  if (alg != INDIGO_QUERY_BFS) return kMaxGang;
  return static_cast<long long>(edges) < 6LL * nodes ? 16 : 128;
}

size_t batch_workspace_bytes(const indigo_graph_ref* graphs, const indigo_query* queries, int nqueries)
{
  return workspace_bytes(graphs, queries, nqueries, INDIGO_MAX_SSSP_SOURCES);
}

int batch_gang(int alg, int nodes, int edges)
{
  if (alg < INDIGO_QUERY_BFS || alg > INDIGO_QUERY_PR || nodes < 0 || edges < 0) return 0;
  const long long entries = static_cast<long long>(edges) + nodes;
  const int cap = gang_cap(alg, nodes, edges, false);
  int k = 1;
  while (k < cap && (static_cast<long long>(k) << kGangShift) < entries) k <<= 1;
  return k;
}

namespace {

int gang_for(int alg, int nodes, int edges, int grid) { return std::min(batch_gang(alg, nodes, edges), std::max(1, grid)); }

// Estimated nanoseconds of one query on one workgroup, fitted to batches of
// one query on graphs of 2^10 to 2^18 entries (and not again since BFS, SSSP, PR and,
// most of all, MIS became faster).
double query_cost(const indigo_query& Q, const indigo_graph_ref& G)
{
  const double entries = static_cast<double>(G.edges) + G.nodes;
  switch (Q.alg) {
    case INDIGO_QUERY_BFS: return entries * 16;
    case INDIGO_QUERY_SSSP: return entries * 7 * Q.nsrc;
    case INDIGO_QUERY_PR: return entries * 35;
    case INDIGO_QUERY_MIS: return entries * 9;
    default: return entries * 5;
  }
}

// Fewest CSR entries per member of a widened gang.  On sparse graphs a BFS or
// SSSP of few sources has levels too narrow to pay a gang barrier for (one BFS
// on a 64^2 grid 0.74 ms on one workgroup, 0.90 on four; 64 at once 4.5 and
// 1.9): the floor is 16 / nsrc times as high for BFS below 16 sources, four
// times for SSSP below 4.
long long widen_floor(const indigo_query& Q, const indigo_graph_ref& G)
{
  if (G.edges < 6LL * G.nodes) {
    if (Q.alg == INDIGO_QUERY_BFS && Q.nsrc < 16) return kWidenEntries * 16 / Q.nsrc;
    if (Q.alg == INDIGO_QUERY_SSSP && Q.nsrc < 4) return kWidenEntries * 4;
  }
  return kWidenEntries;
}

// A batch whose gangs leave workgroups of the grid without a task: the task
// that would finish last (largest cost per member) doubles its gang, while
// the free workgroups last and its members keep widen_floor entries each
// (and the algorithm's bound on gangs holds).  Gangs that a caller chose stay.
// With gangs of 2^18 entries per member alone, a batch was as long as its
// largest task on a workgroup or two (SSSP of 16 sources on 10^5 vertices: 20
// to 30 ms) while most of the grid idled.  Batches of 24, 12, 6 and 2 graphs of
// 2^10 to 2^17 vertices, five algorithms each (at the time of that step): 52.6, 69.5,
// 27.6 and 22.9 -> 15.2, 11.8, 10.8 and 5.0 ms; floors of 1024 and 2048 entries per member
// measured the same within 12%, 16384 up to 23% slower.
void widen_gangs(std::vector<int>& gang, const indigo_graph_ref* graphs, const indigo_query* queries, int grid)
{
  long long used = 0;
  for (int k : gang) used += k;
  if (used >= grid) return;
  using Entry = std::pair<double, int>;  // cost per member, query
  std::priority_queue<Entry> heap;
  for (size_t q = 0; q < gang.size(); q++)
    if (queries[q].gang == 0) heap.push({query_cost(queries[q], graphs[queries[q].graph]) / gang[q], static_cast<int>(q)});
  while (!heap.empty()) {
    const Entry top = heap.top();
    heap.pop();
    const int q = top.second;
    const indigo_graph_ref& G = graphs[queries[q].graph];
    const long long entries = static_cast<long long>(G.edges) + G.nodes;
    const int k = gang[q];
    if (2 * k > gang_cap(queries[q].alg, G.nodes, G.edges, true) || entries / (2 * k) < widen_floor(queries[q], G)) continue;
    if (used + k > grid) continue;
    gang[q] = 2 * k;
    used += k;
    heap.push({top.first / 2, q});
  }
}

}  // namespace

// Workgroups that every persistent kernel of the library can hold resident
// at once: the batch kernel's occupancy with one workgroup per CU left out,
// as for the kernels of more than 80 scalar registers (BFS, SSSP, PageRank
// stop at 3 x 512 threads per CU), so that shares of it assemble side by
// side whatever kernels the sharers run.
int batch_grid_limit(indigo_ctx* ctx, int* limit)
{
  int per_cu = 0;
  IG_TRY(resident_per_cu(ctx, reinterpret_cast<const void*>(batch_kernel), kBatchBlock, 0, &per_cu, false));
  *limit = std::max(1, per_cu * ctx->compute_units);
  return INDIGO_OK;
}

// (Re)launches the batch recorded in ctx->pending_batch; records the stop
// event without waiting.
static int launch_pending(indigo_ctx* ctx)
{
  BatchTask* d_tasks = static_cast<BatchTask*>(ctx->pending_batch.tasks);
  GangState* gangs = static_cast<GangState*>(ctx->pending_batch.gangs);
  BatchControl* ctl = static_cast<BatchControl*>(ctx->pending_batch.ctl);
  int ntasks = ctx->pending_batch.ntasks;
  long long budget = budget_ticks(ctx);
  long long res_ticks = residency_ticks(ctx);
  IG_TRY(timing_begin(ctx));
  IG_TRY(zero_async(ctx, ctl, sizeof(BatchControl)));
  IG_TRY(zero_async(ctx, gangs, static_cast<size_t>(ntasks) * sizeof(GangState)));
  void* args[] = {&d_tasks, &ntasks, &gangs, &ctl, &budget, &res_ticks};
  IG_TRY(coop_launch(ctx, reinterpret_cast<const void*>(batch_kernel), kBatchBlock, 0, args,
                     ctx->pending_batch.grid_cap, nullptr, "batch_kernel", true));
  return timing_record_stop(ctx);
}

int batch_launch(indigo_ctx* ctx, const indigo_graph_ref* graphs, int ngraphs, const indigo_query* queries,
                 int nqueries, int max_workgroups)
{
  if (ctx->pending_batch.active) return set_error(INDIGO_ERR_INVALID_ARG, "batch: the context has a batch in flight");
  if (nqueries < 0 || ngraphs < 0 || (nqueries > 0 && (graphs == nullptr || queries == nullptr)))
    return set_error(INDIGO_ERR_INVALID_ARG, "batch: bad graph / query table");
  if (max_workgroups < 0) return set_error(INDIGO_ERR_INVALID_ARG, "batch: max_workgroups < 0");
  if (nqueries == 0) {
    // an empty batch completes at once: record a stop event for batch_ready
    IG_TRY(timing_begin(ctx));
    IG_TRY(timing_record_stop(ctx));
    ctx->pending_batch = {};
    ctx->pending_batch.active = true;
    return INDIGO_OK;
  }
  for (int g = 0; g < ngraphs; g++) {
    const indigo_graph_ref& G = graphs[g];
    IG_TRY(check_graph_args(G.nodes, G.edges, G.d_nindex, G.d_nlist));
  }
  for (int q = 0; q < nqueries; q++) {
    const indigo_query& Q = queries[q];
    if (Q.graph < 0 || Q.graph >= ngraphs) return set_error(INDIGO_ERR_INVALID_ARG, "batch: query %d graph out of range", q);
    const indigo_graph_ref& G = graphs[Q.graph];
    if (Q.d_out == nullptr) return set_error(INDIGO_ERR_INVALID_ARG, "batch: query %d output is NULL", q);
    if (Q.alg == INDIGO_QUERY_BFS || Q.alg == INDIGO_QUERY_SSSP) {
      const int cap = Q.alg == INDIGO_QUERY_BFS ? INDIGO_MAX_BFS_SOURCES : INDIGO_MAX_SSSP_SOURCES;
      if (Q.nsrc < 1 || Q.nsrc > cap)
        return set_error(INDIGO_ERR_INVALID_ARG, "batch: query %d needs 1..%d sources (got %d)", q, cap, Q.nsrc);
      for (int i = 0; i < Q.nsrc; i++)
        if (Q.src[i] < 0 || Q.src[i] >= G.nodes)
          return set_error(INDIGO_ERR_INVALID_ARG, "batch: query %d source %d out of range", q, Q.src[i]);
      if (Q.alg == INDIGO_QUERY_SSSP && G.d_eweight == nullptr && G.edges > 0)
        return set_error(INDIGO_ERR_INVALID_ARG, "batch: query %d is SSSP on a graph without weights", q);
    } else if (Q.alg != INDIGO_QUERY_CC && Q.alg != INDIGO_QUERY_MIS && Q.alg != INDIGO_QUERY_PR) {
      return set_error(INDIGO_ERR_INVALID_ARG, "batch: query %d has unknown algorithm %d", q, Q.alg);
    }
    if (Q.gang < 0 || Q.gang > kMaxGang)
      return set_error(INDIGO_ERR_INVALID_ARG, "batch: query %d gang %d outside 0..%d", q, Q.gang, kMaxGang);
  }
  // grid: occupancy x CUs (capped), learned residency caps as for the other persistent kernels
  int per_cu = 0;
  IG_TRY(resident_per_cu(ctx, reinterpret_cast<const void*>(batch_kernel), kBatchBlock, 0, &per_cu, true));
  const int grid_cap = std::max(1, max_workgroups > 0 ? std::min(max_workgroups, per_cu * ctx->compute_units)
                                                      : per_cu * ctx->compute_units);
  // tasks, largest gang and work first
  std::vector<int> order(static_cast<size_t>(nqueries));
  std::vector<long long> work(static_cast<size_t>(nqueries));
  for (int q = 0; q < nqueries; q++) {
    order[q] = q;
    const indigo_graph_ref& G = graphs[queries[q].graph];
    work[q] = static_cast<long long>(G.edges) + G.nodes;
  }
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return work[a] > work[b]; });
  std::vector<int> gang(static_cast<size_t>(nqueries));
  for (int q = 0; q < nqueries; q++) {
    const indigo_graph_ref& G = graphs[queries[q].graph];
    gang[q] = queries[q].gang > 0 ? std::min(queries[q].gang, grid_cap)
                                  : gang_for(queries[q].alg, G.nodes, G.edges, grid_cap);
  }
  widen_gangs(gang, graphs, queries, grid_cap);
  const size_t n = static_cast<size_t>(nqueries);
  // SSSPs of several sources take passes of half as many while their rows do not
  // fit the memory (one source a pass needs 20 bytes a vertex)
  int most = INDIGO_MAX_SSSP_SOURCES;
  for (;;) {
    const int rc = ensure_workspace(ctx, workspace_bytes(graphs, queries, nqueries, most));
    if (rc == INDIGO_OK) break;
    if (rc != INDIGO_ERR_OUT_OF_MEMORY || most == 1) return rc;
    clear_error();
    most /= 2;
  }
  IG_TRY(ensure_host_pinned(ctx, n * sizeof(BatchTask)));
  Carver cv(ctx->ws);
  BatchControl* ctl = cv.take<BatchControl>(1);
  GangState* gangs = cv.take<GangState>(n);
  BatchTask* d_tasks = cv.take<BatchTask>(n);
  unsigned char* scratch = cv.take<unsigned char>(0);
  BatchTask* h_tasks = static_cast<BatchTask*>(ctx->host_pinned);
  size_t off = 0;
  for (size_t i = 0; i < n; i++) {
    const indigo_query& Q = queries[order[i]];
    const indigo_graph_ref& G = graphs[Q.graph];
    BatchTask& T = h_tasks[i];
    std::memset(&T, 0, sizeof(T));
    T.alg = Q.alg;
    T.gang = gang[order[i]];
    T.nodes = G.nodes;
    T.edges = G.edges;
    T.rows = pass_rows(Q, most);
    T.item = item_entries(Q.alg, T.rows);
    T.nindex = G.d_nindex;
    T.nlist = G.d_nlist;
    T.eweight = G.d_eweight;
    T.out = Q.d_out;
    T.scratch = scratch + off;
    T.items = reinterpret_cast<int2*>(scratch + off + alg_bytes(Q.alg, G.nodes, G.edges, T.rows));
    off += scratch_bytes(Q.alg, G.nodes, G.edges, T.rows);
    T.nsrc = (Q.alg == INDIGO_QUERY_BFS || Q.alg == INDIGO_QUERY_SSSP) ? Q.nsrc : 0;
    for (int s = 0; s < T.nsrc; s++) T.src[s] = Q.src[s];
  }
  IG_HIP_TRY(hipMemcpyAsync(d_tasks, h_tasks, n * sizeof(BatchTask), hipMemcpyHostToDevice, ctx->stream));
  ctx->pending_batch.active = true;
  ctx->pending_batch.tasks = d_tasks;
  ctx->pending_batch.gangs = gangs;
  ctx->pending_batch.ctl = ctl;
  ctx->pending_batch.ntasks = nqueries;
  ctx->pending_batch.grid_cap = grid_cap;
  return launch_pending(ctx);
}

int batch_ready(indigo_ctx* ctx, int* ready)
{
  if (!ctx->pending_batch.active) return set_error(INDIGO_ERR_INVALID_ARG, "batch: nothing in flight");
  const hipError_t e = hipEventQuery(ctx->ev_stop);
  if (e == hipErrorNotReady) {
    *ready = 0;
    return INDIGO_OK;
  }
  IG_HIP_TRY(e);
  *ready = 1;
  return INDIGO_OK;
}

int batch_wait(indigo_ctx* ctx)
{
  if (!ctx->pending_batch.active) return set_error(INDIGO_ERR_INVALID_ARG, "batch: nothing in flight");
  for (;;) {
    const int ntasks = ctx->pending_batch.ntasks;
    if (ntasks > 0) {
      BatchControl* ctl = static_cast<BatchControl*>(ctx->pending_batch.ctl);
      IG_HIP_TRY(hipMemcpyAsync(ctx->host_pinned, &ctl->bar.abort.v, sizeof(unsigned), hipMemcpyDeviceToHost,
                                ctx->stream));
      IG_HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    const int rc0 = timing_finish(ctx, 3, ntasks);
    if (rc0 != INDIGO_OK || ntasks == 0) {
      ctx->pending_batch.active = false;
      return rc0;
    }
    const unsigned abort_code = *static_cast<unsigned*>(ctx->host_pinned);
    const int rc = check_abort(ctx, reinterpret_cast<const void*>(batch_kernel), abort_code, "batch");
    if (rc != kNotResident) {
      ctx->pending_batch.active = false;
      return rc;
    }
    // the grid did not assemble: relaunch with the lowered residency cap (the
    // device copy of the task table is intact)
    const int lrc = launch_pending(ctx);
    if (lrc != INDIGO_OK) {
      ctx->pending_batch.active = false;
      return lrc;
    }
  }
}

int batch_run(indigo_ctx* ctx, const indigo_graph_ref* graphs, int ngraphs, const indigo_query* queries,
              int nqueries, int max_workgroups)
{
  const int rc = batch_launch(ctx, graphs, ngraphs, queries, nqueries, max_workgroups);
  if (rc == INDIGO_ERR_OUT_OF_MEMORY && nqueries > 1) {
    // the queries' scratch does not fit beside their outputs: half of them at a time
    clear_error();
    const int half = nqueries / 2;
    IG_TRY(batch_run(ctx, graphs, ngraphs, queries, half, max_workgroups));
    const float ms = ctx->last_ms;
    IG_TRY(batch_run(ctx, graphs, ngraphs, queries + half, nqueries - half, max_workgroups));
    ctx->last_ms += ms;
    ctx->last_kernel_ms += ms;
    ctx->last_iterations = nqueries;
    return INDIGO_OK;
  }
  IG_TRY(rc);
  return batch_wait(ctx);
}

}  // namespace indigo
