// Host-side check of the far piles' rotation (csrc/far_piles.hpp), built with g++ by
// tests/test_far_piles.py.
//
// Model: a team enters a phase with an empty near frontier in epoch `entry`, whose pile holds
// something, and runs splits, each of which consumes its epoch's pile, fills the next one and
// clears one.  A workgroup outside the team reads the entry pile's size, by which it
// chooses whether to go on, and arrives at the barrier; it does so before the phase's split
// k for some k, or, where a split waits for it, before that split.  Whenever it reads, it must
// find what the team found.  And no split may clear a pile that still holds something, or
// fill one that was not cleared.  A rule that never waits does not pass.
// Prints "ok" and exits 0 when every check holds.
#include <cstdio>

#include "far_piles.hpp"

namespace {

using indigo::kPiles;
using indigo::pile_cleared;
using indigo::pile_of;
using indigo::split_waits;

constexpr bool never_waits(int, int) { return false; }

// Runs `splits` splits with the outside workgroup late until before split `late`.
template <typename Waits>
bool reads_alike(int entry, int splits, int late, Waits waits)
{
  int size[kPiles] = {0, 0, 0};
  bool live[kPiles] = {false, false, false};  // filled and not yet consumed
  size[pile_of(entry)] = 100 + entry;
  live[pile_of(entry)] = true;
  // consumed by the split before the phase
  size[pile_of(entry + 2)] = 99 + entry;
  const int found = size[pile_of(entry)];
  int read = -1;
  for (int k = 0; k < splits; k++) {
    const int e = entry + k;
    if (read < 0 && (k >= late || waits(entry, e))) read = size[pile_of(entry)];
    if (live[pile_cleared(e)]) return false;
    size[pile_cleared(e)] = 0;
    if (!live[pile_of(e)]) return false;
    live[pile_of(e)] = false;
    if (k > 0 || entry > 1) {
      if (pile_of(e + 1) == pile_of(e) || pile_of(e + 1) == pile_cleared(e)) return false;
      if (k > 0 && size[pile_of(e + 1)] != 0) return false;  // cleared by the split before
    }
    size[pile_of(e + 1)] = 101 + e;
    live[pile_of(e + 1)] = true;
  }
  if (read < 0) read = size[pile_of(entry)];
  return read == found;
}

template <typename Waits>
int failures(Waits waits)
{
  int bad = 0;
  for (int entry = 1; entry < 8; entry++)
    for (int splits = 0; splits < 9; splits++)
      for (int late = 0; late <= splits; late++)
        if (!reads_alike(entry, splits, late, waits)) bad++;
  return bad;
}

}  // namespace

int main()
{
  if (failures(never_waits) == 0) {
    std::fprintf(stderr, "the model does not show the fault of a phase that never waits\n");
    return 1;
  }
  const int bad = failures(split_waits);
  if (bad != 0) {
    std::fprintf(stderr, "%d orders in which a workgroup reads another size\n", bad);
    return 1;
  }
  // one wait a phase
  for (int entry = 1; entry < 8; entry++) {
    int waits = 0;
    for (int e = entry; e < entry + 20; e++) waits += split_waits(entry, e) ? 1 : 0;
    if (waits != 1) return 1;
  }
  std::printf("ok\n");
  return 0;
}
