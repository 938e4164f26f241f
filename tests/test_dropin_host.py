"""The host side of the drop-in penalty calls on stand-ins for the HIP runtime (tests/native/dropin_host_check.c)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("device", ["device", "nodevice"])
def test_penalty_calls(device, tmp_path):
    """Ids that are all out of range need no device, no lock and no message; the others are counted once each."""
    exe = str(tmp_path / "dropin_host_check")
    host = os.path.join(ROOT, "diskllm_amd", "csrc", "host")
    subprocess.run(["gcc", "-O2", "-std=gnu11", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "include"),
                    "-I/opt/rocm/include", "-o", exe, os.path.join(ROOT, "tests", "native", "dropin_host_check.c"),
                    os.path.join(host, "dropin_sampler.c"), os.path.join(host, "dropin_ctx.c"), "-lpthread"], check=True)
    r = subprocess.run([exe, device], capture_output=True, text=True, timeout=60)
    assert r.stdout == "ok\n" and r.stderr == "", r.stdout + r.stderr
