// Stop mark of a loop whose iterations hold one workgroup barrier, as plain code
// (no HIP calls), so that it can be checked on the host without a GPU.
//
// The leader marks an iteration before its barrier, every wave looks after it.  A
// wave may be late with that look: by then the leader may have marked the next
// iteration, but, with the next barrier still ahead of the late wave, no later one.  So the
// mark is the iteration's number and not a flag: a wave that took the next iteration's
// flag for its own would leave the loop alone, and its barriers would meet others of
// the remaining waves.
#pragma once

namespace indigo {

struct PhaseStop {
  int marked;  // iteration at which the loop is left (-1: none)
  constexpr void clear() { marked = -1; }
  constexpr void post(int it, bool stop)
  {
    if (stop) marked = it;
  }
  constexpr bool at(int it) const { return marked == it; }
};

}  // namespace indigo
