"""Host-side check of the rotation of SSSP's far piles (csrc/far_piles.hpp): a
workgroup that is late to read how much a pile holds, while a team already runs
splits, finds what the others found.
tests/far_piles_check.cpp holds the model; it is compiled with g++ (no GPU)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "parallelization-artifact-sc23_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
def test_late_workgroups_read_the_same_pile(tmp_path):
    exe = tmp_path / "far_piles_check"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I" + CSRC,
                           os.path.join(ROOT, "tests", "far_piles_check.cpp"), "-o", str(exe)])
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip() == "ok"


def test_the_kernel_rotates_by_the_checked_rule():
    """Every pile index comes from the header, and the split that clears the entry's
    pile waits before it does."""
    with open(os.path.join(CSRC, "sssp.hip")) as f:
        text = f.read()
    assert re.search(r"far\w*\[[^\]]*% 3", text) is None
    wait = text.index("split_waits(entry, epoch - 1)")
    clear = text.index("far_cnt[pile_cleared(epoch - 1)]")
    assert wait < clear and "wait_others(" in text[wait:clear]
