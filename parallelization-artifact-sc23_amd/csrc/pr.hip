// PageRank (FP32 scores, FP64 convergence test) on gfx950.
//
// Reference semantics: PR_GPU (include/pr_cuda.h:48; constants :42-45) with the
// Jacobi pull of codes/cuda/pr-cuda/PR_CUDA_Pull_FloatType_NonPersist_Thread_
// Determ_GlobalAdd.cu:41-69,91-106: contrib[u] = s[u] / deg[u];
// s'[v] = (1 - 0.85) / N + 0.85 * sum_{u in N(v)} contrib[u]; repeat while the
// L1 change of the iteration is > 1e-4 and fewer than 100 iterations ran.
//
// Design: one persistent kernel; per iteration
//   vertices with short lists (< kPrWaveDeg entries) are taken 64 to a wave (fewer
//   on graphs that would leave waves idle) in vertex order (coalesced score / contrib / index traffic), one lane or one
//   group of lanes to a list;
//   longer lists, collected once into a static list, one wave each; lists of
//   kPrHugeDeg or more in kPrHugeChunk-entry items, one wave each, whose
//   partial sums go to a per-item slot; the wave that finishes a huge
//   vertex's last item (a counter per vertex, and per 32 items) combines its item partials in
//   item order, so no second barrier is needed;
// then one barrier and the stop test.  Per-vertex sums are FP32 with Neumaier
// compensation (the improved Kahan-Babuska sum: a running error term added
// once at the end); wave and workgroup partials are combined pairwise with the
// same error-free step.  contrib is double-buffered and written by the vertex
// that owns it in the pass that computes its score (Jacobi, as the
// reference's Determ variants), so no separate contrib sweep runs.
// |s' - s| is exact in FP64 and summed in FP64, the only FP64 work: each
// workgroup stores its partials in slots (double-buffered by iteration
// parity); after the barrier every workgroup adds all slots in one fixed
// order, so all compute the bit-identical total and take the same stop
// decision (no floating-point atomics).
#include "pr.hpp"

#include <map>
#include <string>
#include <vector>

#include "device_common.hpp"
#include "csum.hpp"
#include "frontier.hpp"
#include "gather.hpp"
#include "trace.hpp"

namespace indigo {

namespace {

constexpr int kPrBlock = 512;
constexpr int kPrHugeDeg = 4096;   // lists split into items
constexpr int kPrHugeChunk = 1024;  // entries per item, one wave each
constexpr int kPrFly = 4;           // items' partials in flight per lane that combines them
constexpr int kPrGroupItems = 32;  // of a vertex's items, counted together
constexpr int kPrBuckets = 16;      // items are ordered by their first neighbour's part of the ids
constexpr float kDamp = 0.85f;

constexpr int kPrMaxGrid = kMaxGraphGrid;  // slots of one workgroup each

// Lists of kPrWaveDeg entries up to kPrHugeDeg by length: class c holds those of
// kPrWaveDeg << c entries up to twice as many.
constexpr int kPrClasses = __builtin_ctz(kPrHugeDeg / kPrWaveDeg);
static_assert(kPrWaveDeg << kPrClasses == kPrHugeDeg, "the classes cover the lists between short and huge");
constexpr int kPrClassCap = 512;  // lists of a class that a workgroup buffers while collecting

struct PrControl {
  GridBarrier bar;
  FrontierCounters heavy;
  PaddedU32 nclass[kPrClasses];
  PaddedU32 nbucket[kPrBuckets];
  int iterations;
  int status;
  double last_diff;
  int grid;
  int pad[25];
  // workgroup 0's timeline: entries 0-2 the end of the set-up (scores,
  // heavy lists, first barrier); then per sweep the start and the ends of its
  // huge, mid and short phases (entry 3 + 4 (it - 1) + phase, mode = phase)
  LevelTrace trace;
};

struct PrArgs {
  int nodes;
  int init_uniform;
  int max_iter;
  double eps;
  const int* __restrict__ nindex;
  const int* __restrict__ nlist;
  const int* __restrict__ degree;  // optional caller-provided degrees (PR_GPU contract)
  float* scores;
  float* contrib[2];
  int* mid[kPrClasses];  // lists of kPrWaveDeg entries and more, by class
  FrontierQueues heavy;  // lists of kPrHugeDeg entries and more (huge)
  unsigned long long* items;  // huge items by bucket (HugeItem, in two words)
  float2* hpart;         // per slot: compensated partial (sum, error)
  int hcap;              // huge vertices at most: edges / kPrHugeDeg + 1
  unsigned* hdone;       // per huge vertex: items (of more than kPrGroupItems, groups of them) finished this sweep
  PaddedU32* gdone;      // per group of items: those finished this sweep
  int ngroups;
  double* hres[2];       // per huge vertex: |s' - s| of a sweep, by its parity: whoever
                         // is late to add them up may see the next sweep's items done
  double* partial;       // [2][2 * kPrMaxGrid] per-workgroup residuals (phase A, phase B)
  int* exit_it;     // [kPrMaxGrid] iteration at which each workgroup left
  double* exit_total;
  PrControl* ctl;
  long long budget;
  long long start_ticks;
};

IG_DEV int deg_of(const PrArgs& a, int v)
{
  return a.degree ? a.degree[v] : a.nindex[v + 1] - a.nindex[v];
}

// New score of v from its gathered sum and its old score; writes score and next
// contrib and returns |s' - s| in FP64.
IG_DEV double finish_vertex(const PrArgs& a, int v, float old, float total, float base, float* cout)
{
  const float s = base + kDamp * total;
  a.scores[v] = s;
  cout[v] = s / static_cast<float>(deg_of(a, v));
  return fabs(static_cast<double>(s) - static_cast<double>(old));
}

IG_DEV void st_float2(float2* p, float2 v)
{
  unsigned long long bits;
  __builtin_memcpy(&bits, &v, sizeof(bits));
  st_relaxed(reinterpret_cast<unsigned long long*>(p), bits);
}

IG_DEV float2 ld_float2(const float2* p)
{
  const unsigned long long bits = ld_relaxed(reinterpret_cast<const unsigned long long*>(p));
  float2 v;
  __builtin_memcpy(&v, &bits, sizeof(v));
  return v;
}

// FP64 sum of one value per thread; result valid in every thread.
IG_DEV double block_sum_f64(double x, double* s_red)
{
  x = wave_sum(x);
  const int wid = threadIdx.x / kWave;
  if (lane_id() == 0) s_red[wid] = x;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < kPrBlock / kWave; w++) t += s_red[w];
  __syncthreads();
  return t;
}

// Part of the list of huge vertex number j: entries [beg, end), partial in slot.
struct HugeItem {
  int j, slot, beg, end;
};

// First group of huge vertex number j, whose slots start at first: the numbers and the slots
// of the vertices rise together, so no two vertices share a group.
IG_DEV int group_of(int first, int j) { return first / kPrGroupItems + j; }

// Items of huge vertex v.
IG_DEV int huge_items(const PrArgs& a, int v)
{
  return static_cast<int>((static_cast<unsigned>(a.nindex[v + 1] - a.nindex[v]) + kPrHugeChunk - 1u) / kPrHugeChunk);
}

// Item k of huge vertex number j, which is v and whose slots start at first.
IG_DEV HugeItem huge_item(const PrArgs& a, int j, unsigned first, int k, int v)
{
  const int beg = a.nindex[v] + k * kPrHugeChunk, end = a.nindex[v + 1];
  return {j, static_cast<int>(first) + k, beg, end - beg < kPrHugeChunk ? end : beg + kPrHugeChunk};
}

// Counts a finished item of a vertex with `items` of them, whose slots start at first;
// whether it was the sweep's last.  One counter took the 1024 items of a list of 2^20
// entries one after the other (a star's call 2.52 -> 2.10 ms with groups).
IG_DEV bool item_done(const PrArgs& a, const HugeItem& item, int first, int items)
{
  if (items <= kPrGroupItems) return atomic_add_relaxed(&a.hdone[item.j], 1u) + 1u == static_cast<unsigned>(items);
  const int g = (item.slot - first) / kPrGroupItems, groups = (items + kPrGroupItems - 1) / kPrGroupItems;
  const int members = min(kPrGroupItems, items - g * kPrGroupItems);
  unsigned* group = &a.gdone[group_of(first, item.j) + g].v;
  if (atomic_add_relaxed(group, 1u) + 1u != static_cast<unsigned>(members)) return false;
  st_relaxed(group, 0u);
  return atomic_add_relaxed(&a.hdone[item.j], 1u) + 1u == static_cast<unsigned>(groups);
}

IG_DEV unsigned long long pack(int lo, int hi)
{
  return static_cast<unsigned long long>(static_cast<unsigned>(hi)) << 32 | static_cast<unsigned>(lo);
}

IG_DEV void unpack(unsigned long long x, int& lo, int& hi)
{
  lo = static_cast<int>(x);
  hi = static_cast<int>(x >> 32);
}

__global__ __launch_bounds__(kPrBlock) void pr_kernel(PrArgs a)
{
  __shared__ double s_red[kPrBlock / kWave];
  __shared__ unsigned s_bucket[kPrBuckets], s_slot[kPrBuckets];
  __shared__ FrontierEmitterT<64, 64, 64> s_emit;
  __shared__ BlockQueue<kPrClassCap> s_class[kPrClasses];
  __shared__ unsigned s_nclass[kPrClasses];
  PrControl* ctl = a.ctl;
  if (!residency_barrier(&ctl->bar, a.start_ticks)) return;
  const long long deadline = now_ticks() + a.budget;
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  const int stride = gridDim.x * blockDim.x;
  const int lane = lane_id();
  const int wpb = kPrBlock / kWave;
  const float inv_n = 1.0f / static_cast<float>(a.nodes);
  const float base = (1.0f - kDamp) / static_cast<float>(a.nodes);

  const int wave = static_cast<int>(blockIdx.x) * wpb + static_cast<int>(threadIdx.x) / kWave;
  const int nwaves = static_cast<int>(gridDim.x) * wpb;
  // A wave's place among the waves moves on by about 4/9 of them a turn.  On R-MAT
  // graphs a list's length goes with the set bits of its vertex id, so a wave that
  // kept its place, a multiple of 2^11 vertices apart, met the same kind of
  // lists every turn (R-MAT 22: 7.06 ms a call, 6.6 with the moves).
  const int move = (nwaves * 4 / 9) & ~(wpb - 1);
  auto next_turn = [&](int at) { return at + move < nwaves ? at + move : at + move - nwaves; };

  if (tid == 0) ctl->trace.start = now_ticks();
  for (int v = tid; v < a.nodes; v += stride) {
    const float s = a.init_uniform ? inv_n : a.scores[v];
    a.scores[v] = s;
    a.contrib[0][v] = s / static_cast<float>(deg_of(a, v));
  }
  for (int j = tid; j < a.hcap; j += stride) st_relaxed(&a.hdone[j], 0u);
  for (int g = tid; g < a.ngroups; g += stride) st_relaxed(&a.gdone[g].v, 0u);
  trace_level(&ctl->trace, 0, 0u, 0ull, 0);
  fe_reset(s_emit);
  for (int c = 0; c < kPrClasses; c++) bq_reset(s_class[c]);
  const int runs = a.nodes / kWave + (a.nodes % kWave != 0 ? 1 : 0);
  for (int w0 = 0, at = wave; w0 < runs; w0 += nwaves, at = next_turn(at)) {
    const int v = (w0 + at) * kWave + lane;
    const int deg = w0 + at < runs && v < a.nodes ? a.nindex[v + 1] - a.nindex[v] : 0;
    if (__ballot(deg >= kPrWaveDeg) == 0ull) continue;
    for (int c = 0; c < kPrClasses; c++)
      bq_append(s_class[c], deg >= kPrWaveDeg << c && deg < kPrWaveDeg << (c + 1), v, a.mid[c], &ctl->nclass[c].v);
    frontier_emit_block<kPrHugeDeg, kPrHugeDeg, kPrHugeChunk>(s_emit, deg >= kPrHugeDeg, v, deg, a.heavy, &ctl->heavy);
  }
  for (int c = 0; c < kPrClasses; c++) bq_flush(s_class[c], a.mid[c], &ctl->nclass[c].v);
  fe_flush(s_emit, a.heavy, &ctl->heavy);
  trace_level(&ctl->trace, 1, 0u, 0ull, 1);
  if (!grid_barrier(&ctl->bar, deadline)) {
    if (tid == 0) ctl->status = 1;
    if (threadIdx.x == 0) a.exit_it[blockIdx.x] = -1000000;
    return;
  }
  trace_level(&ctl->trace, 2, 0u, 0ull, 2);
  if (threadIdx.x < kPrClasses) s_nclass[threadIdx.x] = ld_relaxed(&ctl->nclass[threadIdx.x].v);
  __syncthreads();
  const unsigned long long hp = ld_relaxed(&ctl->heavy.hpack);
  const unsigned nh = huge_count(hp), nch = huge_chunks(hp);

  // Huge items.  While there is one for a wave at most, it keeps it; otherwise they
  // are ordered by where in the ids they begin (counted, then placed), so that at
  // any time the waves gather from one part of the contributions, which the L2s
  // hold, and not from all of them (R-MAT 22, 16 MB: the items' part of a sweep
  // 130 -> 56 us, a call 5.87 -> 5.61 ms; with lists of 1024 entries and more in
  // items 6.0: an item costs three round trips beyond its entries).
  const bool ordered = nch > static_cast<unsigned>(nwaves);
  HugeItem own{};
  if (!ordered && static_cast<unsigned>(wave) < nch) {
    const int j = huge_owner_wave(a.heavy.hoff, static_cast<int>(nh), static_cast<unsigned>(wave));
    const unsigned first = ld_relaxed(&a.heavy.hoff[j]);
    own = huge_item(a, j, first, static_cast<int>(wave - first), ld_relaxed(&a.heavy.hq[j]));
  }
  for (int pass = 0; ordered && pass < 2; pass++) {
    if (threadIdx.x < kPrBuckets) s_bucket[threadIdx.x] = 0u;
    __syncthreads();
    for (unsigned j = static_cast<unsigned>(wave); j < nh; j += nwaves) {
      const int v = ld_relaxed(&a.heavy.hq[j]);
      const unsigned first = ld_relaxed(&a.heavy.hoff[j]);
      const int items = huge_items(a, v);
      for (int k = lane; k < items; k += kWave) {
        const HugeItem item = huge_item(a, static_cast<int>(j), first, k, v);
        const unsigned b = static_cast<unsigned>(static_cast<unsigned long long>(a.nlist[item.beg]) * kPrBuckets /
                                                 static_cast<unsigned>(a.nodes));
        const unsigned n = atomicAdd(&s_bucket[b], 1u);
        if (pass == 1) {
          st_relaxed(&a.items[2 * (s_slot[b] + n)], pack(item.j, item.slot));
          st_relaxed(&a.items[2 * (s_slot[b] + n) + 1], pack(item.beg, item.end));
        }
      }
    }
    __syncthreads();
    if (pass == 0 && threadIdx.x < kPrBuckets)
      s_slot[threadIdx.x] = atomic_add_relaxed(&ctl->nbucket[threadIdx.x].v, s_bucket[threadIdx.x]);
    if (!grid_barrier<true>(&ctl->bar, deadline)) {
      if (tid == 0) ctl->status = 1;
      if (threadIdx.x == 0) a.exit_it[blockIdx.x] = -1000000;
      return;
    }
    if (pass == 0 && threadIdx.x < kPrBuckets)
      for (unsigned b = 0; b < threadIdx.x; b++) s_slot[threadIdx.x] += ld_relaxed(&ctl->nbucket[b].v);
  }

  // mid lists, the longest first, are dealt to the workgroups in turn, and to
  // their waves in turn: by class, the shares differ by less than a list of each
  // (unsorted, the workgroups finished a sweep of R-MAT 22 after 660 to 910 us).
  // This wave's first list is number rest0 of class c0.
  auto next_list = [&](unsigned& c, unsigned& rest) {
    while (c > 0 && rest >= s_nclass[c]) rest -= s_nclass[c--];
    return rest < s_nclass[c];
  };
  unsigned c0 = kPrClasses - 1;
  unsigned rest0 = threadIdx.x / kWave * gridDim.x + blockIdx.x;
  const bool has_mid = next_list(c0, rest0);
  // short lists: vertices per wave and turn (fewer while waves are free,
  // where lists average enough entries for the groups)
  int per = kWave;
  const bool dense = a.nindex[a.nodes] >= kPrLaneDeg * static_cast<long long>(a.nodes);
  const int least = dense ? kWave / kPrGroup : kWave;
  while (per > least && (a.nodes + per / 2 - 1) / (per / 2) <= nwaves) per /= 2;
  const int chunks = (a.nodes + per - 1) / per;
  const bool few = per <= kWave / kPrGroup;

  int it = 0;
  for (;;) {
    it++;
    const float* cin = a.contrib[(it - 1) & 1];
    float* cout = a.contrib[it & 1];
    auto contribution = [cin](int u) { return cin[u]; };
    double* slots = a.partial + (it & 1) * (2 * kPrMaxGrid);
    double d = 0.0;
    const int tl = 3 + 4 * (it - 1);
    trace_level(&ctl->trace, tl, static_cast<unsigned>(it), 0ull, 0);

    // huge items -> partials; the last item of a vertex combines them
    for (unsigned p = static_cast<unsigned>(wave); p < nch; p += nwaves) {
      HugeItem item = own;
      if (ordered) {
        unpack(ld_relaxed(&a.items[2 * p]), item.j, item.slot);
        unpack(ld_relaxed(&a.items[2 * p + 1]), item.beg, item.end);
      }
      const int v = a.heavy.hq[item.j];  // (in flight beside the gathers)
      const int items = huge_items(a, v);
      const unsigned first = a.heavy.hoff[item.j];
      CSum acc;
      gather<kWave>(acc, contribution, a.nlist, item.beg, item.end, lane);
      acc = wave_merge(acc);
      bool last = false;
      if (lane == 0) {
        // the partial and the counter are device-scope accesses, the store
        // completed before the count (agent-scope acquire / release fences
        // would write back and invalidate the XCD's L2, and with it the
        // cached contributions every gather reads: 6.8 -> 9.7 ms)
        st_float2(&a.hpart[item.slot], make_float2(acc.s, acc.c));
        wave_drain();
        last = item_done(a, item, static_cast<int>(first), items);
      }
      if (__ballot(last) != 0ull) {
        // (kPrFly partials a round trip: a star of 2^20 vertices 2.69 -> 2.52 ms)
        CSum tot;
        for (int q0 = lane; q0 < items; q0 += kPrFly * kWave) {
          float2 part[kPrFly];
#pragma unroll
          for (int q = 0; q < kPrFly; q++) {
            const int k = q0 + q * kWave;
            part[q] = k < items ? ld_float2(&a.hpart[first + k]) : make_float2(0.f, 0.f);
          }
#pragma unroll
          for (int q = 0; q < kPrFly; q++)
            if (q0 + q * kWave < items) tot.merge(part[q].x, part[q].y);
        }
        tot = wave_merge(tot);
        if (lane == 0) {
          st_relaxed(&a.hres[it & 1][item.j], finish_vertex(a, v, a.scores[v], tot.value(), base, cout));
          st_relaxed(&a.hdone[item.j], 0u);  // every item of this sweep has counted
        }
      }
    }
    trace_level(&ctl->trace, tl + 1, static_cast<unsigned>(it), 0ull, 1);
    // phase A: mid lists, one wave each
    unsigned c = c0, rest = rest0;
    for (bool more = has_mid; more; rest += nwaves, more = next_list(c, rest)) {
      const int v = a.mid[c][rest];
      const int beg = a.nindex[v], end = a.nindex[v + 1];
      const float old = a.scores[v];
      CSum acc;
      gather<kWave>(acc, contribution, a.nlist, beg, end, lane);
      acc = wave_merge(acc);
      if (lane == 0) d += finish_vertex(a, v, old, acc.value(), base, cout);
    }
    trace_level(&ctl->trace, tl + 2, static_cast<unsigned>(it), 0ull, 2);
    // phase A: short lists, `per` vertices a wave, vertex order
    for (int c0 = 0, at = wave; c0 < chunks; c0 += nwaves, at = next_turn(at)) {
      const int c = c0 + at;
      const int v = c * per + lane;
      const bool mine = lane < per && c < chunks && v < a.nodes;
      const int beg = mine ? a.nindex[v] : 0, end = mine ? a.nindex[v + 1] : 0;
      const float old = mine ? a.scores[v] : 0.f;  // (in flight beside the gathers)
      const float sum = short_sums(contribution, a.nlist, beg, end, few);
      if (mine && end - beg < kPrWaveDeg) d += finish_vertex(a, v, old, sum, base, cout);
    }
    d = block_sum_f64(d, s_red);
    if (threadIdx.x == 0) slots[2 * blockIdx.x] = d;
    d = 0.0;
    trace_level(&ctl->trace, tl + 3, static_cast<unsigned>(it), 0ull, 3);

    if (!grid_barrier(&ctl->bar, deadline)) {
      if (tid == 0) ctl->status = 1;
      if (threadIdx.x == 0) a.exit_it[blockIdx.x] = -it;
      return;
    }
    // every workgroup adds all slots, then the huge vertices' residuals, in
    // one fixed order: the same total everywhere, whichever workgroup
    // combined which huge vertex
    double part = 0.0;
    for (int b = threadIdx.x; b < static_cast<int>(gridDim.x); b += kPrBlock) part += slots[2 * b];
    double hpart_sum = 0.0;
    for (int j = threadIdx.x; j < static_cast<int>(nh); j += kPrBlock) hpart_sum += ld_relaxed(&a.hres[it & 1][j]);
    const double total = block_sum_f64(part, s_red) + block_sum_f64(hpart_sum, s_red);
    if (!(total > a.eps && it < a.max_iter)) {
      if (tid == 0) {
        ctl->iterations = it;
        ctl->last_diff = total;
        ctl->grid = gridDim.x;
      }
      if (threadIdx.x == 0) {
        a.exit_it[blockIdx.x] = it;
        a.exit_total[blockIdx.x] = total;
      }
      break;
    }
  }
}

}  // namespace

// Upper bound on the number of huge items: every huge list has at least
// kPrHugeDeg entries, so items <= edges / kPrHugeChunk + edges / kPrHugeDeg.
static size_t pr_max_chunks(int edges)
{
  return static_cast<size_t>(edges) / kPrHugeChunk + static_cast<size_t>(edges) / kPrHugeDeg + 2;
}

// Groups of items at most: the last vertex's begin at pr_max_chunks / kPrGroupItems + its number
// at most.
static size_t pr_max_groups(int edges)
{
  return pr_max_chunks(edges) / kPrGroupItems + static_cast<size_t>(edges) / kPrHugeDeg + 2;
}

// Lists of class c at most.
static size_t pr_class_cap(int edges, int c) { return static_cast<size_t>(edges) / (kPrWaveDeg << c) + 1; }

size_t pr_workspace_bytes(int nodes, int edges)
{
  const size_t v = static_cast<size_t>(nodes);
  size_t mid = 0;
  for (int c = 0; c < kPrClasses; c++) mid += Carver::round(pr_class_cap(edges, c) * 4);
  return Carver::round(sizeof(PrControl)) + mid + 5 * Carver::round(v * 4) + Carver::round(pr_max_chunks(edges) * 16) +
         Carver::round(pr_max_chunks(edges) * 8) +
         Carver::round((static_cast<size_t>(edges) / kPrHugeDeg + 1) * 20) + 512 +
         Carver::round(pr_max_groups(edges) * sizeof(PaddedU32)) +
         Carver::round(4 * kPrMaxGrid * 8) + Carver::round(kPrMaxGrid * 4) + Carver::round(kPrMaxGrid * 8) + 4096;
}

// Workgroups of one call, per square root of the entries.  Measured on R-MAT 12, 14,
// 16 and 18 (0.1M to 7.6M entries) the best caps were 64, 128, 256 and 512 (calls
// 0.31 -> 0.15, 0.35 -> 0.19, 0.45 -> 0.31 and 0.69 -> 0.64 ms); from about 2^25
// entries on the rule exceeds the resident grid, which is kept.
constexpr double kPrGridPerRoot = 0.2;

int pr_run(indigo_ctx* ctx, int nodes, int edges, const int* nindex, const int* nlist, const int* degree,
           float* scores, int init_uniform)
{
  Carver cv(ctx->ws);
  PrArgs a{};
  a.ctl = cv.take<PrControl>(1);
  a.contrib[0] = cv.take<float>(nodes);
  a.contrib[1] = cv.take<float>(nodes);
  a.heavy.q = nullptr;
  a.heavy.mq = nullptr;
  for (int c = 0; c < kPrClasses; c++) a.mid[c] = cv.take<int>(pr_class_cap(edges, c));
  a.heavy.hq = cv.take<int>(nodes);
  a.heavy.hoff = cv.take<unsigned>(nodes);
  a.items = cv.take<unsigned long long>(2 * pr_max_chunks(edges));
  a.hpart = cv.take<float2>(pr_max_chunks(edges));
  a.hcap = edges / kPrHugeDeg + 1;  // every huge list holds kPrHugeDeg entries or more
  a.hdone = cv.take<unsigned>(static_cast<size_t>(a.hcap));
  a.ngroups = static_cast<int>(pr_max_groups(edges));
  a.gdone = cv.take<PaddedU32>(static_cast<size_t>(a.ngroups));
  for (double*& hres : a.hres) hres = cv.take<double>(static_cast<size_t>(a.hcap));
  a.partial = cv.take<double>(4 * kPrMaxGrid);
  a.exit_it = cv.take<int>(kPrMaxGrid);
  a.exit_total = cv.take<double>(kPrMaxGrid);
  ctx->diag[0] = a.exit_it;
  ctx->diag[1] = a.exit_total;
  a.nodes = nodes;
  a.init_uniform = init_uniform;
  a.max_iter = 100;
  a.eps = static_cast<double>(0.0001f);
  a.nindex = nindex;
  a.nlist = nlist;
  a.degree = degree;
  a.scores = scores;
  a.budget = budget_ticks(ctx);
  a.start_ticks = residency_ticks(ctx);
  IG_TRY(zero_async(ctx, a.ctl, sizeof(PrControl)));
  IG_TRY(zero_async(ctx, a.exit_it, sizeof(int) * kPrMaxGrid));
  void* args[] = {&a};
  IG_TRY(coop_launch(ctx, reinterpret_cast<const void*>(pr_kernel), kPrBlock, 0, args,
                     graph_grid(nodes, edges, kPrGridPerRoot), nullptr, "pr_kernel"));
  return INDIGO_OK;
}

int pr_collect(indigo_ctx* ctx, int* iterations, double* last_diff)
{
  Carver cv(ctx->ws);
  PrControl* ctl = cv.take<PrControl>(1);
  IG_TRY(ensure_host_pinned(ctx, sizeof(PrControl)));
  PrControl* h = static_cast<PrControl*>(ctx->host_pinned);
  IG_HIP_TRY(hipMemcpyAsync(h, ctl, sizeof(PrControl), hipMemcpyDeviceToHost, ctx->stream));
  IG_HIP_TRY(hipStreamSynchronize(ctx->stream));
  IG_TRY(check_abort(ctx, reinterpret_cast<const void*>(pr_kernel), h->bar.abort.v, "pagerank"));
  if (h->status != 0) {
    // which iteration each workgroup left at (negative: its barrier gave
    // up), and the stop total it computed
    const int g = kPrMaxGrid;
    std::vector<int> it(g);
    std::vector<double> tot(g);
    IG_HIP_TRY(hipMemcpy(it.data(), ctx->diag[0], sizeof(int) * g, hipMemcpyDeviceToHost));
    IG_HIP_TRY(hipMemcpy(tot.data(), ctx->diag[1], sizeof(double) * g, hipMemcpyDeviceToHost));
    std::map<int, int> by_it;
    std::map<double, int> by_total;
    for (int b = 0; b < g; b++) {
      if (it[b] == 0) continue;
      by_it[it[b]]++;
      if (it[b] > 0) by_total[tot[b]]++;
    }
    std::string msg;
    for (auto& kv : by_it) msg += " it" + std::to_string(kv.first) + "x" + std::to_string(kv.second);
    msg += " | totals:";
    int shown = 0;
    for (auto& kv : by_total) {
      if (shown++ == 6) break;
      char buf[64];
      snprintf(buf, sizeof(buf), " %.17g x%d", kv.first, kv.second);
      msg += buf;
    }
    char bar[160];
    snprintf(bar, sizeof(bar), " | barrier groups %u %u %u %u %u %u %u %u top %u gen %u",
             h->bar.group[0].v, h->bar.group[1].v, h->bar.group[2].v, h->bar.group[3].v, h->bar.group[4].v,
             h->bar.group[5].v, h->bar.group[6].v, h->bar.group[7].v, h->bar.top.v, h->bar.gen.v);
    msg += bar;
    msg += " | grid " + std::to_string(ctx->last_grid) + " per_cu " + std::to_string(ctx->last_per_cu) + " cus " +
           std::to_string(ctx->compute_units);
    return set_error(INDIGO_ERR_TIMEOUT, "pagerank: persistent kernel stopped (status %d); workgroups:%s",
                     h->status, msg.c_str());
  }
  store_trace(ctx, h->trace);
  if (iterations) *iterations = h->iterations;
  if (last_diff) *last_diff = h->last_diff;
  return INDIGO_OK;
}

}  // namespace indigo
