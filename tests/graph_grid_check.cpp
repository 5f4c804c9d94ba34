// Host-side check of the grid sizes chosen from a graph (graph_grid in
// csrc/grid_plan.hpp), built with g++ by tests/test_graph_grid.py.  Prints "ok" and
// exits 0 when every check holds.
#include <climits>
#include <cstdio>

#include "grid_plan.hpp"

using indigo::graph_grid;

static int failures = 0;

static void check(int nodes, int edges, double per_root, int want)
{
  const int got = graph_grid(nodes, edges, per_root);
  if (got == want) return;
  std::fprintf(stderr, "graph_grid(%d, %d, %g) = %d, expected %d\n", nodes, edges, per_root, got, want);
  failures++;
}

int main()
{
  // by the entries, as long as they are 1.5 for a vertex or more
  check(1 << 12, 1 << 17, 0.2, 64);
  check(1 << 14, 1 << 19, 0.2, 128);
  check(1 << 16, 1 << 21, 0.2, 256);
  check(1 << 16, 1 << 21, 0.4, 512);
  check(1 << 20, 3 << 19, 0.2, 256);
  check(1 << 22, 128 << 20, 0.2, 2048);
  // many vertices, few entries or none
  check(1 << 24, 1 << 16, 0.2, 1024);
  check(1 << 24, 0, 0.2, 1024);
  check(1 << 24, 1 << 16, 0.4, 2048);
  check(1 << 22, 1 << 12, 0.2, 512);
  check(1 << 20, 1 << 16, 0.2, 256);
  check(1 << 18, 1 << 10, 0.2, 128);
  check(1 << 16, 1 << 10, 0.2, 64);
  // bounds, and the rounding: up from sqrt(2) times a power of two on
  check(1, 0, 0.2, 64);
  check(1, INT_MAX, 0.4, indigo::kMaxGraphGrid);
  check(INT_MAX, 0, 0.4, indigo::kMaxGraphGrid);
  check(INT_MAX, INT_MAX, 1e9, indigo::kMaxGraphGrid);
  check(1, 204799, 0.2, 64);
  check(1, 204801, 0.2, 128);
  // never fewer workgroups for more vertices or more entries
  for (int v = 1; v < 1 << 25; v = v * 3 / 2 + 1)
    for (int e = 0; e < 1 << 28; e = e * 3 / 2 + 1) {
      const int g = graph_grid(v, e, 0.2);
      if (g < 64 || g > indigo::kMaxGraphGrid || graph_grid(v, e + 1, 0.2) < g || graph_grid(v + 1, e, 0.2) < g) {
        std::fprintf(stderr, "graph_grid(%d, %d) not monotonic or out of range\n", v, e);
        failures++;
      }
    }
  if (failures == 0) std::printf("ok\n");
  return failures == 0 ? 0 : 1;
}
