"""Host-side check of the grids that BFS, MIS and PageRank choose by a graph's size
(csrc/grid_plan.hpp): by its entries, or by its vertices where these are the work.
tests/graph_grid_check.cpp holds the cases; it is compiled with g++ (no GPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "parallelization-artifact-sc23_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
def test_grids_by_graph_size(tmp_path):
    exe = tmp_path / "graph_grid_check"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I" + CSRC,
                           os.path.join(ROOT, "tests", "graph_grid_check.cpp"), "-o", str(exe)])
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip() == "ok"
