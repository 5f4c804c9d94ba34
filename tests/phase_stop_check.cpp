// Host-side check of a phase loop's stop mark (csrc/phase_stop.hpp), built with
// g++ by tests/test_phase_stop.py.
//
// Model of the loop: the leader marks iteration i when it should end (it looks on every second, fourth, ...
// iteration), the barrier of iteration i follows, then the leader and a late wave each
// look whether iteration i is marked and leave when it is.  The late wave looks either
// before or after the leader has gone on and marked iteration i + 1; it is
// past neither that iteration's barrier nor the leader's.  Every choice of early
// and late looks over the iterations is taken, and both must leave in the iteration
// that was marked.  A flag that all iterations share does not pass.
// Prints "ok" and exits 0 when every check holds.
#include <cstdio>

#include "phase_stop.hpp"

namespace {

struct OneFlag {
  int flag;
  void clear() { flag = 0; }
  void post(int, bool stop) { flag = stop ? 1 : 0; }
  bool at(int) const { return flag != 0; }
};

// Runs iterations first .. first + n - 1, posting every `period`, with the stop due at
// iteration `stop`; bit i of `late` delays the wave's read of iteration first + i
// past the leader's next post.  True when both leave at `stop`.
template <typename Flag>
bool leave_together(int first, int n, int period, int stop, unsigned late)
{
  Flag f{};
  f.clear();
  int leader_left = -1, wave_left = -1;
  auto post = [&](int it) {
    if (it % period == 0) f.post(it, it >= stop);
  };
  post(first);
  for (int i = 0; i < n && leader_left < 0 && wave_left < 0; i++) {
    const int it = first + i;  // (the barrier of `it`)
    if (f.at(it)) leader_left = it;
    const bool is_late = (late >> i & 1u) != 0u && leader_left < 0;
    if (!is_late && f.at(it)) wave_left = it;
    if (leader_left < 0) post(it + 1);
    if (is_late && f.at(it)) wave_left = it;
  }
  return leader_left == stop && wave_left == stop;
}

template <typename Flag>
int failures()
{
  int bad = 0;
  for (int first = 0; first < 8; first++)
    for (int period = 2; period <= 8; period *= 2)
      for (int n = 2; n <= 10; n++) {
        const int stop = (first + n - 1) / period * period;
        if (stop < first) continue;
        for (unsigned late = 0; late < 1u << n; late++)
          if (!leave_together<Flag>(first, n, period, stop, late)) bad++;
      }
  return bad;
}

}  // namespace

int main()
{
  if (failures<OneFlag>() == 0) {
    std::fprintf(stderr, "the model does not show a shared flag's fault\n");
    return 1;
  }
  const int bad = failures<indigo::PhaseStop>();
  if (bad != 0) {
    std::fprintf(stderr, "%d interleavings in which a wave leaves alone\n", bad);
    return 1;
  }
  std::printf("ok\n");
  return 0;
}
