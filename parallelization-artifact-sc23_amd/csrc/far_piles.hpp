// SSSP's far piles: three buffers, by epoch, as plain arithmetic (no HIP calls), so
// that their use can be checked on the host without a GPU.
#pragma once

namespace indigo {

constexpr int kPiles = 3;

// The pile of an epoch.
constexpr int pile_of(int epoch) { return epoch % kPiles; }

// The pile that the split from epoch to epoch + 1 clears: consumed by the split before, it
// is filled from the next split on.
constexpr int pile_cleared(int epoch) { return (epoch + 2) % kPiles; }

// A team phase that was entered with an empty near frontier in epoch `entry` runs splits
// while workgroups outside the team may still be about to read how much that epoch's
// pile holds, by which they choose the pass.  Whether the split from `epoch` is the first to
// clear that pile, before which all of them have to have arrived at the barrier.
constexpr bool split_waits(int entry, int epoch) { return epoch == entry + 1; }

}  // namespace indigo
