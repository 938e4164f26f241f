"""The receipt validator's transition table against its scanner, on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_receipt_table_is_the_scanner(tmp_path):
    exe = str(tmp_path / "receipt_table_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "include"),
                    "-I/opt/rocm/include", "-o", exe, os.path.join(ROOT, "tests", "native", "receipt_table_check.cpp")],
                   check=True)
    states, checked, bad = map(int, subprocess.run([exe], capture_output=True, text=True, timeout=120).stdout.split())
    assert states == 70 and checked > 1000000 and bad == 0
