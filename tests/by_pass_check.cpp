// Host-side check of the values that a team phase leaves for the grid (csrc/by_pass.hpp),
// built with g++ by tests/test_by_pass.py.
//
// Model: passes 0 .. n - 1, each of them a phase (one workgroup runs it and stores
// 1000 + R before the pass's barrier) or a pass of the whole grid (nothing stored).
// After a phase's barrier a second workgroup reads the value; it does so at once, or only
// when the first has gone through the next pass up to its barrier, which it cannot pass
// without the second.  Over every mix of passes and every choice of late reads the
// second must find what the phase before stored.  One slot does not pass.
// Prints "ok" and exits 0 when every check holds.
#include <cstdio>

#include "by_pass.hpp"

namespace {

struct OneSlot {
  int slot;
  int& of(int) { return slot; }
};

template <typename Slots>
bool all_read_their_own(int n, unsigned phases, unsigned late)
{
  Slots s{};
  bool ok = true;
  auto run = [&](int R) {
    if (phases >> R & 1u) s.of(R) = 1000 + R;
  };
  run(0);
  for (int R = 0; R < n; R++) {  // (the barrier of pass R)
    const bool is_late = (late >> R & 1u) != 0u;
    const bool reads = (phases >> R & 1u) != 0u;
    if (reads && !is_late) ok = ok && s.of(R) == 1000 + R;
    if (R + 1 < n) run(R + 1);
    if (reads && is_late) ok = ok && s.of(R) == 1000 + R;
  }
  return ok;
}

template <typename Slots>
int failures()
{
  int bad = 0;
  for (int n = 1; n <= 8; n++)
    for (unsigned phases = 0; phases < 1u << n; phases++)
      for (unsigned late = 0; late < 1u << n; late++)
        if (!all_read_their_own<Slots>(n, phases, late)) bad++;
  return bad;
}

}  // namespace

int main()
{
  if (failures<OneSlot>() == 0) {
    std::fprintf(stderr, "the model does not show a single slot's fault\n");
    return 1;
  }
  const int bad = failures<indigo::ByPass<int>>();
  if (bad != 0) {
    std::fprintf(stderr, "%d orders in which a workgroup reads another pass's value\n", bad);
    return 1;
  }
  std::printf("ok\n");
  return 0;
}
