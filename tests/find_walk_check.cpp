// Host-side check of the union-find walk (csrc/find_walk.hpp), built with g++ by
// tests/test_find_walk.py.
//
// All finds of a tree run in lockstep, as a GPU's lanes do: in each step, every find
// that is still under way makes one load, in id order.  The starting trees are those
// of cc_init: a chain, and the chains of a mesh with ids row by row (each vertex under
// the smallest of its neighbours).
// Every find must return the root, parents must stay ancestors, and the number
// of steps must stay far below the walk that stores nothing on its way (kMark 0), which on
// a chain of n takes more than sqrt(n).  A tree no deeper than kDepth gets no store.
// Prints "ok" and exits 0 when every check holds.
#include <ucontext.h>

#include <cstdio>
#include <utility>
#include <vector>

#include "find_walk.hpp"

namespace {

constexpr int kDepth = 5, kMark = 64;  // as in unionfind.hpp
constexpr size_t kStack = 16384;

int failures = 0;

void check(bool ok, const char* what, long long got)
{
  if (ok) return;
  std::fprintf(stderr, "%s (%lld)\n", what, got);
  failures++;
}

struct Run {
  std::vector<int> parent;
  std::vector<int> found;
  std::vector<ucontext_t> fiber;
  std::vector<char> stacks;
  ucontext_t main;
  long long stores = 0;
  bool marks = false;
  int at = 0;

  int load(int v)
  {
    swapcontext(&fiber[at], &main);  // the step's one load follows the switch back
    return parent[v];
  }
  void store(int v, int p)
  {
    check(p < parent[v] || (p == parent[v] && p < v), "a store that is no ancestor", v);
    parent[v] = p;
    stores++;
  }
};

Run* g_run;

void body()
{
  Run& r = *g_run;
  const int x = r.at;
  auto load = [&r](int v) { return r.load(v); };
  auto store = [&r](int v, int p) { r.store(v, p); };
  r.found[x] = r.marks ? indigo::find_walk<kDepth, kMark>(x, load, store) : indigo::find_walk<kDepth, 0>(x, load, store);
}

// Steps until every find has returned.
int lockstep(std::vector<int> parent, bool marks, int root, long long* stores)
{
  Run r;
  g_run = &r;
  const int n = static_cast<int>(parent.size());
  r.parent = std::move(parent);
  r.found.assign(n, -1);
  r.fiber.resize(n);
  r.stacks.resize(kStack * n);
  r.marks = marks;
  for (int v = 0; v < n; v++) {
    getcontext(&r.fiber[v]);
    r.fiber[v].uc_stack.ss_sp = &r.stacks[kStack * v];
    r.fiber[v].uc_stack.ss_size = kStack;
    r.fiber[v].uc_link = &r.main;
    makecontext(&r.fiber[v], body, 0);
  }
  int steps = 0;
  for (int left = n; left > 0; steps++) {
    left = 0;
    for (int v = 0; v < n; v++) {
      if (r.found[v] >= 0) continue;
      r.at = v;
      swapcontext(&r.main, &r.fiber[v]);
      if (r.found[v] < 0) left++;
    }
  }
  for (int v = 0; v < n; v++) check(r.found[v] == root, "a find that missed the root", v);
  *stores = r.stores;
  return steps;
}

std::vector<int> chain(int n)
{
  std::vector<int> p(n);
  for (int v = 0; v < n; v++) p[v] = v > 0 ? v - 1 : 0;
  return p;
}

std::vector<int> mesh(int rows, int cols)
{
  std::vector<int> p(rows * cols);
  for (int v = 0; v < rows * cols; v++) p[v] = v >= cols ? v - cols : (v > 0 ? v - 1 : 0);
  return p;
}

}  // namespace

int main()
{
  long long s0 = 0, s1 = 0;
  // allowed: the kMark hops up to the first mark, then two steps for each doubling of the reach
  for (int n : {1, 2, 5, 6, 7, 63, 64, 65, 129, 4096, 8192, 16384}) {
    const int plain = lockstep(chain(n), false, 0, &s0), marked = lockstep(chain(n), true, 0, &s1);
    int log2n = 0;
    while ((1 << log2n) < n) log2n++;
    check(marked <= kMark + 2 * log2n + 2, "a chain's finds take too many steps", marked);
    if (n >= 8192) check(plain > kMark + 2 * log2n + 2, "the model does not show an unmarked chain's walks", plain);
    std::printf("chain %d: %d steps without marks, %d with\n", n, plain, marked);
    if (n <= kDepth + 1) check(s1 == 0, "a store into a shallow tree", s1);
  }
  for (int rows : {16, 1024}) {
    const int cols = 16384 / rows;
    const int plain = lockstep(mesh(rows, cols), false, 0, &s0), marked = lockstep(mesh(rows, cols), true, 0, &s1);
    check(marked <= plain, "a mesh's finds take longer with marks", marked);
    std::printf("mesh %d x %d: %d steps without marks, %d with\n", rows, cols, plain, marked);
  }
  if (failures == 0) std::printf("ok\n");
  return failures == 0 ? 0 : 1;
}
