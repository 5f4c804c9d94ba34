// Degree-binned frontier queues for the persistent traversal kernels.
//
// Queue contents and counters are written and read with device-scope atomic
// accesses only, so kernels built on them may use the coherent grid barrier.
//
// A frontier is three queues, binned by adjacency-list length when a vertex
// is appended:
//   * small: length < kMidDeg.  Expanded 64 vertices per wave with an in-wave
//     load balancer (prefix sum of lengths + owner search), so a wave always
//     handles 64 consecutive CSR entries and never more than 64 * 63 in all;
//   * mid:   kMidDeg <= length < kHugeDeg.  One wave per vertex (several
//     while there are few), lanes striding its list (coalesced);
//   * huge:  length >= kHugeDeg.  Split into kHugeChunk-entry work items, one
//     wave each.  Its counter packs (chunk count << 32 | vertex count) so one
//     64-bit atomic allocates both the slots and the vertices' first chunk
//     indices; hoff[] is therefore sorted by slot and a wave finds a chunk's
//     owner by a 64-way search.
// kHugeDeg bounds a wave's serial chain to 8 windows of about 3 us.  With lists
// of up to 4095 entries on one wave (and longer ones in 2048-entry workgroup
// items), the longest list set an iteration: SSSP on R-MAT 22, 20, 18 and 16
// took 4.95, 2.11, 0.91 and 0.66 ms, now 4.09, 1.43, 0.76 and 0.50.
// Appends are aggregated by wave (ballot + mbcnt prefix, one atomic per wave and
// queue) or, in the passes of the whole grid, by workgroup (emit.hpp).  Counters are triple-buffered across levels so that the set written
// in level L, read in L+1 and cleared in L+2 never has two roles at once.
//
// The same machinery bins a static vertex set: collect_heavy() appends every
// vertex of length >= kMidDeg of a graph to the mid / huge queues, while the
// short lists are walked in vertex-id order (coalesced) by the kernels.
#pragma once

#include "device_common.hpp"
#include "emit.hpp"

namespace indigo {

constexpr int kMidDeg = 64;
constexpr int kHugeDeg = 512;
constexpr int kHugeChunk = 512;

struct alignas(128) FrontierCounters {
  unsigned int n;            // small queue length
  unsigned int nm;           // mid queue length
  unsigned long long hpack;  // (huge chunks << 32) | huge queue length
  unsigned long long m;      // sum of lengths over the frontier
  unsigned long long aux;    // algorithm-specific
  unsigned long long pad[12];
};

// Per-level trace written by workgroup 0 of a traversal kernel: wall-clock
// tick at the start of the level, frontier size, its degree sum and the mode
// (0 top-down, 1 bottom-up, 2 team phase, 3 far-pile split).
constexpr int kTraceMax = 256;
struct LevelTrace {
  int n;
  int pad;
  long long start;
  long long t[kTraceMax];
  unsigned nf[kTraceMax];
  unsigned long long m[kTraceMax];
  int mode[kTraceMax];
};

IG_DEV void trace_level(LevelTrace* tr, int level, unsigned nf, unsigned long long m, int mode)
{
  if (blockIdx.x == 0 && threadIdx.x == 0 && level < kTraceMax) {
    tr->t[level] = now_ticks();
    tr->nf[level] = nf;
    tr->m[level] = m;
    tr->mode[level] = mode;
    tr->n = level + 1;
  }
}

struct FrontierQueues {
  int* q;          // small queue
  int* mq;         // mid queue
  int* hq;         // huge queue
  unsigned* hoff;  // first chunk index of each huge entry
};

IG_DEV unsigned huge_count(unsigned long long hpack) { return static_cast<unsigned>(hpack & 0xffffffffull); }
IG_DEV unsigned huge_chunks(unsigned long long hpack) { return static_cast<unsigned>(hpack >> 32); }

IG_DEV void counters_clear(FrontierCounters* c)
{
  st_relaxed(&c->n, 0u);
  st_relaxed(&c->nm, 0u);
  st_relaxed(&c->hpack, 0ull);
  st_relaxed(&c->m, 0ull);
  st_relaxed(&c->aux, 0ull);
}

// Snapshot of a counter set (device-scope loads).
IG_DEV FrontierCounters counters_load(const FrontierCounters* c)
{
  FrontierCounters r;
  r.n = ld_relaxed(&c->n);
  r.nm = ld_relaxed(&c->nm);
  r.hpack = ld_relaxed(&c->hpack);
  r.m = ld_relaxed(&c->m);
  r.aux = ld_relaxed(&c->aux);
  return r;
}

// First chunk indices of a wave's huge vertices, appended straight to the global
// queue with one atomic (all lanes converged).
template <int kChunk>
IG_DEV void huge_append(bool huge, int u, int deg, const FrontierQueues& fq, FrontierCounters* c)
{
  const unsigned long long hm = __ballot(huge);
  if (hm == 0) return;
  const int chunks = huge ? (deg + kChunk - 1) / kChunk : 0;
  const int incl = wave_inclusive_scan(chunks);
  const int total = wave_shfl(incl, kWave - 1);
  const int leader = __ffsll(static_cast<long long>(hm)) - 1;
  unsigned long long old = 0;
  if (lane_id() == leader)
    old = atomic_add_relaxed(&c->hpack, (static_cast<unsigned long long>(total) << 32) | __popcll(hm));
  old = wave_shfl(old, leader);
  if (huge) {
    const unsigned slot = static_cast<unsigned>(old & 0xffffffffull) + lanes_below(hm);
    st_relaxed(&fq.hq[slot], u);
    st_relaxed(&fq.hoff[slot], static_cast<unsigned>(old >> 32) + static_cast<unsigned>(incl - chunks));
  }
}

// Wave-collective: every active lane with `pred` appends vertex u (whose list
// has deg entries) to the frontier `fq`/`c`.  All 64 lanes must be converged.
IG_DEV void frontier_emit(bool pred, int u, int deg, const FrontierQueues& fq, FrontierCounters* c)
{
  const bool huge = pred && deg >= kHugeDeg;
  const bool mid = pred && deg >= kMidDeg && !huge;
  const bool small = pred && deg < kMidDeg;
  const unsigned long long dsum = wave_sum(static_cast<unsigned long long>(pred ? deg : 0));
  if (lane_id() == 0 && dsum != 0) atomic_add_relaxed(&c->m, dsum);
  wave_append(small, u, fq.q, &c->n);
  wave_append(mid, u, fq.mq, &c->nm);
  huge_append<kHugeChunk>(huge, u, deg, fq, c);
}

// Workgroup-aggregated version of frontier_emit (see emit.hpp): appends and the
// degree sum are buffered in LDS and flushed with one atomic per queue by
// fe_flush.  A huge entry takes its slot and its first chunk index from one
// 64-bit LDS atomic, so both stay sorted; entries beyond kHugeCap go straight to
// the global queue.
constexpr int kEmitSmallCap = 4096;
constexpr int kEmitMidCap = 512;
constexpr int kEmitHugeCap = 256;

template <int kSmallCap, int kMidCap, int kHugeCap>
struct FrontierEmitterT {
  BlockQueue<kSmallCap> small;
  BlockQueue<kMidCap> mid;
  BlockSum m;
  unsigned long long hpack;  // (chunks << 32) | buffered huge entries
  unsigned long long hbase;  // the same of the global queue before this workgroup's
  int hu[kHugeCap];
  unsigned hchunk[kHugeCap];
};
using FrontierEmitter = FrontierEmitterT<kEmitSmallCap, kEmitMidCap, kEmitHugeCap>;
// For collect_heavy over a whole graph with a low threshold: no small queue,
// room for a workgroup's whole share of mid lists (an append beyond the
// buffer costs a same-address global atomic, about 10 ns each, serialised).
using HeavyCollector = FrontierEmitterT<64, 2048, 64>;

// Workgroup-collective.
template <int S, int M, int H>
IG_DEV void fe_reset(FrontierEmitterT<S, M, H>& E)
{
  if (threadIdx.x == 0) {
    E.small.count = 0;
    E.mid.count = 0;
    E.m.v = 0ull;
    E.hpack = 0ull;
  }
  __syncthreads();
}

// Wave-collective.  kMid and kHuge are the list lengths from which a vertex
// goes to the mid and the huge queue, kChunk the entries per huge chunk.
template <int kMid = kMidDeg, int kHuge = kHugeDeg, int kChunk = kHugeChunk, int S, int M, int H>
IG_DEV void frontier_emit_block(FrontierEmitterT<S, M, H>& E, bool pred, int u, int deg, const FrontierQueues& fq,
                                FrontierCounters* c)
{
  if (__ballot(pred) == 0ull) return;
  const bool huge = pred && deg >= kHuge;
  const bool mid = pred && deg >= kMid && !huge;
  const bool small = pred && deg < kMid;
  bs_add(E.m, static_cast<unsigned long long>(pred ? deg : 0));
  bq_append(E.small, small, u, fq.q, &c->n);
  bq_append(E.mid, mid, u, fq.mq, &c->nm);
  const unsigned long long hm = __ballot(huge);
  if (hm == 0) return;
  const int chunks = huge ? (deg + kChunk - 1) / kChunk : 0;
  const int incl = wave_inclusive_scan(chunks);
  const int total = wave_bcast(incl, kWave - 1);
  const int pop = __popcll(hm);
  const int leader = __ffsll(static_cast<long long>(hm)) - 1;
  unsigned long long old = 0;
  int room = 0;
  if (lane_id() == leader) {
    // taken only while the whole batch fits, so that the buffered entries
    // are a gapless prefix
    old = E.hpack;
    for (;;) {
      room = static_cast<int>(old & 0xffffffffull) + pop <= H;
      if (!room) break;
      const unsigned long long got =
          atomicCAS(&E.hpack, old, old + ((static_cast<unsigned long long>(total) << 32) | static_cast<unsigned>(pop)));
      if (got == old) break;
      old = got;
    }
  }
  room = wave_shfl(room, leader);
  if (room == 0) {
    huge_append<kChunk>(huge, u, deg, fq, c);
    return;
  }
  old = wave_shfl(old, leader);
  if (huge) {
    const int slot = static_cast<int>(old & 0xffffffffull) + lanes_below(hm);
    E.hu[slot] = u;
    E.hchunk[slot] = static_cast<unsigned>(old >> 32) + static_cast<unsigned>(incl - chunks);
  }
}

// Workgroup-collective.
template <int S, int M, int H>
IG_DEV void fe_flush(FrontierEmitterT<S, M, H>& E, const FrontierQueues& fq, FrontierCounters* c)
{
  __syncthreads();
  const int nh = static_cast<int>(E.hpack & 0xffffffffull);
  if (nh > 0) {
    if (threadIdx.x == 0) E.hbase = atomic_add_relaxed(&c->hpack, E.hpack);
    __syncthreads();
    const unsigned slot0 = static_cast<unsigned>(E.hbase & 0xffffffffull);
    const unsigned chunk0 = static_cast<unsigned>(E.hbase >> 32);
    for (int i = threadIdx.x; i < nh; i += blockDim.x) {
      st_relaxed(&fq.hq[slot0 + i], E.hu[i]);
      st_relaxed(&fq.hoff[slot0 + i], chunk0 + E.hchunk[i]);
    }
  }
  bq_flush(E.small, fq.q, &c->n);
  bq_flush(E.mid, fq.mq, &c->nm);
  if (threadIdx.x == 0 && E.m.v != 0ull) atomic_add_relaxed(&c->m, E.m.v);
  __syncthreads();
}

// Index j of the huge entry owning chunk `item`: the last j with hoff[j] <= item.
IG_DEV int huge_owner(const unsigned* hoff, int nh, unsigned item)
{
  int lo = 0, hi = nh - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (ld_relaxed(&hoff[mid]) <= item) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// The same, by a whole wave (all lanes converged): 64 probes a step, so two
// dependent loads for up to 4096 huge entries.
IG_DEV int huge_owner_wave(const unsigned* hoff, int nh, unsigned item)
{
  int lo = 0, n = nh;  // the answer is in [lo, lo + n)
  while (n > 1) {
    const int step = (n + kWave - 1) / kWave;
    const int at = lane_id() * step;
    // lane 0's probe holds (its entry starts at or before item), the others
    // hold up to the answer's own block
    const unsigned long long le = __ballot(at < n && (at == 0 || ld_relaxed(&hoff[lo + at]) <= item));
    const int block = __popcll(le) - 1;
    lo += block * step;
    n = min(step, n - block * step);
  }
  return lo;
}

// Workgroup-collective grid-stride pass over vertices 0..nodes-1 (64 per
// wave) that appends every vertex with a list of >= kMid entries to the mid /
// huge queues, aggregated per workgroup.
template <int kMid, int kHuge, int kChunk, int S, int M, int H>
IG_DEV void collect_heavy(FrontierEmitterT<S, M, H>& E, int nodes, const int* __restrict__ nindex,
                          const FrontierQueues& fq, FrontierCounters* c)
{
  const int lane = lane_id();
  const int wpb = blockDim.x / kWave;
  const int nw = (nodes + kWave - 1) / kWave;
  fe_reset(E);
  for (int w = blockIdx.x * wpb + threadIdx.x / kWave; w < nw; w += gridDim.x * wpb) {
    const int v = w * kWave + lane;
    const int deg = v < nodes ? nindex[v + 1] - nindex[v] : 0;
    frontier_emit_block<kMid, kHuge, kChunk>(E, deg >= kMid, v, deg, fq, c);
  }
  fe_flush(E, fq, c);
}

// ---- expansion helpers ------------------------------------------------------
// Each calls f(v, e, active) with all lanes of the wave (or all threads of the
// workgroup) converged; `active` says whether (v, e) is a real CSR entry of a
// frontier vertex v.  f may use wave-collective operations.

// Waves per item of a pass over n items on the grid's waves: the largest
// power of two up to `most` that leaves no wave with two items.
IG_DEV unsigned waves_per_item(unsigned n, unsigned most)
{
  const unsigned nwaves = gridDim.x * (blockDim.x / kWave);
  unsigned k = 1;
  while (k < most && static_cast<unsigned long long>(n) * k * 2 <= nwaves) k *= 2;
  return k;
}

// Huge lists: one wave per kHugeChunk-entry item, or, while there are few items,
// k waves each (k up to one per window), wave j taking windows j, j + k, ...
template <typename F>
IG_DEV void expand_huge(const FrontierQueues& in, unsigned nh, unsigned nch, const int* __restrict__ nindex, F&& f)
{
  const int lane = lane_id();
  const unsigned wpb = blockDim.x / kWave;
  const unsigned k = waves_per_item(nch, kHugeChunk / kWave);
  for (unsigned i = blockIdx.x * wpb + threadIdx.x / kWave; i < nch * k; i += gridDim.x * wpb) {
    const unsigned item = i / k;
    const int j = huge_owner_wave(in.hoff, static_cast<int>(nh), item);
    const int v = ld_relaxed(&in.hq[j]);
    const int beg = nindex[v] + static_cast<int>(item - ld_relaxed(&in.hoff[j])) * kHugeChunk;
    const int end = min(nindex[v + 1], beg + kHugeChunk);
    for (int base = beg + static_cast<int>(i % k) * kWave; base < end; base += static_cast<int>(k) * kWave) {
      const int e = base + lane;
      f(v, e, e < end);
    }
  }
}

// Mid lists: one wave each, or, while there are few of them, k waves each (k
// up to one per window), wave j of a list taking its windows j, j + k, ...
// Each window is a chain of device-scope
// round trips (the neighbour's check, its claim or atomicMin, its degree), so a
// 4000-entry list walked by one wave set a level's length: BFS's level of 997
// lists and 3.6M entries on R-MAT 22 took 198 us (calls 0.65 -> 0.53 ms).
template <typename F>
IG_DEV void expand_mid(const FrontierQueues& in, unsigned nm, const int* __restrict__ nindex, F&& f)
{
  const int lane = lane_id();
  const unsigned wpb = blockDim.x / kWave;
  const unsigned k = waves_per_item(nm, kHugeDeg / kWave);
  for (unsigned i = blockIdx.x * wpb + threadIdx.x / kWave; i < nm * k; i += gridDim.x * wpb) {
    const int v = ld_relaxed(&in.mq[i / k]);
    const int beg = nindex[v], end = nindex[v + 1];
    for (int base = beg + static_cast<int>(i % k) * kWave; base < end; base += static_cast<int>(k) * kWave) {
      const int e = base + lane;
      f(v, e, e < end);
    }
  }
}

// Vertices per wave of an expand_small pass over n small-queue vertices of
// average list length `avg`: 64 when they fill the grid's waves, else fewer,
// down to about one 64-entry window per wave.  A wave's windows are serial
// chains of round trips (2 to 3 us each), so 64 vertices of 16 entries on one
// wave made a narrow level 30 to 50 us long while most waves had nothing to
// do; below one window per wave, more workgroups only means more
// same-address appends at the flush.  SSSP calls on R-MAT 12 and 16 0.65 and
// 0.87 -> 0.29 and 0.70 ms, random 2^20 (degree 16) 2.28 -> 1.27, 1024^2 and
// 2048^2 roads 29.8 and 74.2 -> 20.7 and 48.6; BFS on the 2048^2 road 40.3 ->
// 28.4 ms, random 2^20 0.36 -> 0.28.
IG_DEV unsigned small_share(unsigned n, unsigned avg)
{
  const unsigned nwaves = gridDim.x * (blockDim.x / kWave);
  unsigned per = kWave;
  while (per > 1 && per * avg > kWave && (n + per / 2 - 1) / (per / 2) <= nwaves) per /= 2;
  return per;
}

// Small lists: `per` (at most 64) vertices per wave, 64 CSR entries per step.
template <typename F>
IG_DEV void expand_small(const int* __restrict__ q, unsigned n, const int* __restrict__ nindex, F&& f,
                         unsigned per = kWave)
{
  const unsigned lane = lane_id();
  const unsigned wpb = blockDim.x / kWave;
  for (unsigned c = blockIdx.x * wpb + threadIdx.x / kWave; c * per < n; c += gridDim.x * wpb) {
    const unsigned idx = c * per + lane;
    const bool valid = lane < per && idx < n;
    const int v = valid ? ld_relaxed(&q[idx]) : 0;
    const int beg = valid ? nindex[v] : 0;
    const int deg = valid ? nindex[v + 1] - beg : 0;
    const int incl = wave_inclusive_scan(deg);
    const int total = wave_shfl(incl, kWave - 1);
    for (int base = 0; base < total; base += kWave) {
      const int k = base + lane;
      const int o = min(wave_owner(incl, k), kWave - 1);
      const int ov = wave_shfl(v, o);
      const int obeg = wave_shfl(beg, o);
      const int oexcl = wave_shfl(incl - deg, o);
      f(ov, obeg + (k - oexcl), k < total);
    }
  }
}

}  // namespace indigo
