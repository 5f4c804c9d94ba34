// The walk of a union-find's find, as plain code over the caller's load and store
// of parents (no HIP calls), so that its length can be checked on the host
// without a GPU.
//
// A walk stores only into the vertex it started from: the root at its end if it took
// more than kDepth hops, and, where it takes kMark hops (0: never), the ancestor it
// has reached, again each time it has twice as many behind it.  Each store
// replaces the parent of a vertex that is no root by one of its ancestors, so
// concurrent finds and links stay valid.  unionfind.hpp has the reasons.
#pragma once

#include <climits>

namespace indigo {

template <int kDepth, int kMark, typename Load, typename Store>
__attribute__((always_inline)) constexpr int find_walk(int x, Load&& load, Store&& store)
{
  int r = x, p = load(x);
  int hops = 0;
  for (int mark = kMark > 0 ? kMark : INT_MAX;; mark *= 2) {
    while (p != r && hops < mark) {
      r = p;
      p = load(r);
      hops++;
    }
    if (p == r) break;
    store(x, r);
  }
  if (hops > kDepth) store(x, r);
  return r;
}

}  // namespace indigo
