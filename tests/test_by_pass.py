"""Host-side check of what a team phase of BFS and SSSP leaves for the grid
(csrc/by_pass.hpp): a workgroup that is late to read it, while the next phase has
already ended, finds what its own pass left.
tests/by_pass_check.cpp holds the model; it is compiled with g++ (no GPU)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "parallelization-artifact-sc23_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
def test_late_workgroups_read_their_own_pass(tmp_path):
    exe = tmp_path / "by_pass_check"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I" + CSRC,
                           os.path.join(ROOT, "tests", "by_pass_check.cpp"), "-o", str(exe)])
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip() == "ok"


@pytest.mark.parametrize("source,fields", [("bfs.hip", ["level", "last_m"]),
                                           ("sssp.hip", ["it", "split", "epoch", "last_m"])])
def test_team_phases_hand_over_by_pass(source, fields):
    """Each value is stored once and read once, both by the pass."""
    with open(os.path.join(CSRC, source)) as f:
        text = f.read()
    for name in fields:
        assert len(re.findall(r"st_relaxed\(&ctl->base\.of\(R\)\.%s, " % name, text)) == 1
        assert len(re.findall(r"ld_relaxed\(&ctl->base\.of\(R\)\.%s\)" % name, text)) == 1
