"""Host-side check of the union-find walk behind CC (csrc/find_walk.hpp): the finds
of a chain, all under way at once, end after a number of steps that grows with the
logarithm of its length.  tests/find_walk_check.cpp holds the lockstep model; it is
compiled with g++ (no GPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "parallelization-artifact-sc23_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
def test_finds_of_a_chain_in_lockstep(tmp_path):
    exe = tmp_path / "find_walk_check"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I" + CSRC,
                           os.path.join(ROOT, "tests", "find_walk_check.cpp"), "-o", str(exe)])
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip().endswith("ok")
