// PageRank's gathers: compensated sums of a vertex's neighbours' contributions,
// by a lane, a group of lanes, a wave or a workgroup per list.  The loads are the
// caller's (at(u) is the contribution of u): plain ones where a barrier makes the
// last sweep's stores visible, device-scope ones where it does not.
#pragma once

#include "csum.hpp"

namespace indigo {

constexpr int kPrLaneDeg = 8;   // shorter lists: one lane each (twice as long where no list of the wave is longer)
constexpr int kPrWaveDeg = 64;  // longer lists up to this: one group of lanes each
constexpr int kPrGroup = 8;     // lanes of a group
constexpr int kPrUnroll = 4;    // gathers in flight per lane

// acc += at(nlist[e]) for e = beg + first, beg + first + step, ... < end,
// in that order, with kPrUnroll independent loads in flight per lane: the
// gathers are latency-bound chains (index, then contribution), so a plain
// loop would wait out one round trip per window.  Past the end a lane adds 0.
template <int kStep, typename F>
IG_DEV void gather(CSum& acc, F&& at, const int* __restrict__ nlist, int beg, int end, int first)
{
  for (int e = beg + first; e < end; e += kPrUnroll * kStep) {
    int u[kPrUnroll];
#pragma unroll
    for (int q = 0; q < kPrUnroll; q++) u[q] = e + q * kStep < end ? nlist[e + q * kStep] : -1;
    float c[kPrUnroll];
#pragma unroll
    for (int q = 0; q < kPrUnroll; q++) c[q] = u[q] >= 0 ? at(u[q]) : 0.f;
#pragma unroll
    for (int q = 0; q < kPrUnroll; q++) acc.add(c[q]);
  }
}

// Sum over the kPrGroup lanes of a group, in each of them.
IG_DEV CSum group_merge(CSum a)
{
#pragma unroll
  for (int d = kPrGroup / 2; d > 0; d >>= 1) {
    const float s2 = __shfl_xor(a.s, d, kWave);
    const float c2 = __shfl_xor(a.c, d, kWave);
    a.merge(s2, c2);
  }
  return a;
}

// Wave-collective: the gathered sum of each lane's list [beg, end) where it has
// fewer than kPrWaveDeg entries (0 elsewhere).  Lists of fewer than kPrLaneDeg
// entries are summed by their own lane; the others go kPrGroup lanes to a list,
// kWave / kPrGroup lists at a time, instead of a wave to a list of 16 to 63
// (random graph of 2^20 vertices and degree 16: 2.06 -> 1.11 ms a call).  A wave
// without lists of 2 * kPrLaneDeg entries leaves all to their lanes: on degree 4
// the few longer ones' extra step cost 5%.
// few: the wave has at most kWave / kPrGroup lists, all of them grouped.
template <typename F>
IG_DEV float short_sums(F&& at, const int* __restrict__ nlist, int beg, int end, bool few)
{
  const int lane = lane_id();
  const int deg = end - beg;
  const bool any = few || __ballot(deg >= 2 * kPrLaneDeg && deg < kPrWaveDeg) != 0ull;
  const int limit = few ? 1 : (any ? kPrLaneDeg : 2 * kPrLaneDeg);
  CSum own;
  if (deg < limit) gather<1>(own, at, nlist, beg, end, 0);
  float sum = own.value();
  if (!any) return sum;
  const bool grouped = deg >= limit && deg < kPrWaveDeg;
  const unsigned long long m = __ballot(grouped);
  const int rows = __popcll(m);
  const int rank = lanes_below(m);
  // lane r gets (of) the lane of the r-th grouped list (others push past the rows)
  const int rest = lane - rank + rows;  // lanes without a grouped list, in order, behind them
  const int of = __builtin_amdgcn_ds_permute((grouped ? rank : rest) << 2, lane);
  constexpr int kPer = kWave / kPrGroup;
  for (int r0 = 0; r0 < rows; r0 += kPer) {
    const int r = r0 + lane / kPrGroup;
    const int from = wave_shfl(of, r < kWave ? r : kWave - 1);
    const int b = wave_shfl(beg, from), e = wave_shfl(end, from);
    CSum acc;
    if (r < rows) gather<kPrGroup>(acc, at, nlist, b, e, lane % kPrGroup);
    acc = group_merge(acc);
    const float v = wave_shfl(acc.value(), ((rank - r0) & (kPer - 1)) * kPrGroup);
    if (grouped && rank >= r0 && rank < r0 + kPer) sum = v;
  }
  return sum;
}

}  // namespace indigo
