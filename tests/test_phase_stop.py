"""Host-side check of the stop mark that the team phases of BFS and SSSP read
after their one barrier per iteration (csrc/phase_stop.hpp): whichever waves are
late with the read, all leave in the same iteration.
tests/phase_stop_check.cpp holds the model; it is compiled with g++ (no GPU)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "parallelization-artifact-sc23_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
def test_waves_leave_a_phase_together(tmp_path):
    exe = tmp_path / "phase_stop_check"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I" + CSRC,
                           os.path.join(ROOT, "tests", "phase_stop_check.cpp"), "-o", str(exe)])
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip() == "ok"


@pytest.mark.parametrize("source", ["bfs.hip", "sssp.hip"])
def test_team_phases_use_the_checked_flag(source):
    """The kernels post and read through PhaseStop."""
    with open(os.path.join(CSRC, source)) as f:
        text = f.read()
    assert len(re.findall(r"\bstop\.post\(", text)) == 1
    assert len(re.findall(r"\bstop\.at\(", text)) == 1
    assert "abort_flag" not in text
