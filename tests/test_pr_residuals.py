"""Model (CPU) of the stop test of PageRank's sweeps, which every workgroup makes by
itself after the sweep's barrier: it adds the residuals of the split lists, each
stored by whoever finished the list's last item.  A workgroup that is late to add
them up, while others go on to the next sweep up to its barrier, still takes the
same decision, in every order of late reads; with one slot per list it does not.
And the kernel's stores and reads take the checked slot."""
import itertools
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def sweeps_left(residuals, eps, slots, late):
    """The sweeps after which two workgroups stop: the first finishes every list, the
    second, which is late after sweep t where late[t], only adds up.  After the
    barrier of sweep t the first may run all of sweep t + 1."""
    slot = [None] * slots
    stopped = [None, None]
    slot[0] = residuals[0]
    for t in range(len(residuals)):
        i = t % slots
        if not late[t] and not slot[i] > eps:
            stopped[1] = t
        if not slot[i] > eps:
            stopped[0] = t
        elif t + 1 < len(residuals):
            slot[(t + 1) % slots] = residuals[t + 1]
        if late[t] and not slot[i] > eps:
            stopped[1] = t
        if stopped[0] is not None or stopped[1] is not None:
            return stopped
    return stopped


def test_late_workgroups_take_the_same_decision():
    residuals = [0.85 ** t for t in range(9)]
    faults = {1: 0, 2: 0}
    for slots in faults:
        for stop in range(8):
            eps = 0.5 * (residuals[stop] + (residuals[stop - 1] if stop else 2.0))
            for late in itertools.product([False, True], repeat=len(residuals)):
                left = sweeps_left(residuals, eps, slots, late)
                faults[slots] += left != [stop, stop]
    assert faults[2] == 0
    assert faults[1] > 0


def test_the_kernel_takes_the_slot_of_the_sweep():
    with open(os.path.join(ROOT, "parallelization-artifact-sc23_amd", "csrc", "pr.hip")) as f:
        text = f.read()
    uses = re.findall(r"(st|ld)_relaxed\(&a\.hres(\[it & 1\])?\[", text)
    assert sorted(uses) == [("ld", "[it & 1]"), ("st", "[it & 1]")]
