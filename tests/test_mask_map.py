"""The grammar mask kernel's split of rows over blocks: blocks that share a CU are worth it for many rows only."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_rows_are_split_where_it_pays(tmp_path):
    exe = str(tmp_path / "mask_map_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(ROOT, "tests", "native", "mask_map_check.cpp")], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120).stdout
    shapes, wrong, crowded = map(int, out.split())
    assert shapes > 1000000 and wrong == 0 and crowded == 0
