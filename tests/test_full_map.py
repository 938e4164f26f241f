"""The fused kernel's mapping of workgroups to rows and slices: every row of every grid can finish on any number of
XCDs (a workgroup holds its place while it waits for its row's others)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_row_finishes(tmp_path):
    exe = str(tmp_path / "full_map_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(ROOT, "tests", "native", "full_map_check.cpp")], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300).stdout
    grids, stuck, pairs, stuck_pairs, wrong, groups, stuck_groups, stuck_halves = map(int, out.split())
    assert grids > 1500 and pairs > 50 and wrong == 0
    assert stuck == 0 and stuck_pairs == 0
    # grids of several streams; in halves they would get stuck, which is why the host leaves that mapping then
    assert groups == 1350 and stuck_groups == 0 and stuck_halves > 0
