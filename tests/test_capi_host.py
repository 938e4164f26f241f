"""The host side of dlk_sample on stand-ins for the HIP runtime (tests/native/capi_host_check.cpp): what it does with
its workspaces around the kernel launches."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    build = tmp_path_factory.mktemp("capi_host")
    obj, exe = str(build / "capi_host.o"), str(build / "capi_host_check")
    inc = "-I" + os.path.join(ROOT, "include")
    subprocess.run([HIP, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", inc, "-c",
                    os.path.join(ROOT, "diskllm_amd", "csrc", "hip", "capi.hip"), "-o", obj], check=True)
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", inc, "-I/opt/rocm/include", "-o", exe,
                    os.path.join(ROOT, "tests", "native", "capi_host_check.cpp"), obj, "-lpthread",
                    "-Wl,--unresolved-symbols=ignore-in-object-files"], check=True)

    def run(commands):
        r = subprocess.run([exe] + commands.split(), capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout.splitlines()
    return run


FULL, TOPK = "64 151936 151936 0 1.0", "64 128256 128256 40 0.8"


@pytest.mark.parametrize("call,kernel", [(FULL, "fused"), (TOPK, "top-k")])
def test_fresh_workspace_is_cleared_on_the_stream_of_the_call(host, call, kernel):
    """The counters of a fresh workspace are cleared in the order of the call's own stream: a clear on the null stream
    is not waited for by a non-blocking one, and the kernel's row barriers then count from whatever is there."""
    out = host(f"sample {call} 7 sample {call} 7")
    at = [i for i, line in enumerate(out) if "kernel" in line]
    at = [i for i in at if "mapping" not in out[i]]
    assert len(at) == 2 and all(out[i] == f"{kernel} kernel, 64 rows on stream 7" for i in at), out
    assert out[0].startswith("malloc") and out[1] == "clear on stream 7" and at[0] == 2, out
    assert not any("memset" in line for line in out), out
    assert sum("clear" in line for line in out) == 1, out       # the kernels return their counters to zero


@pytest.mark.parametrize("call,history,kernel", [
    # greedy over short rows, of any alignment
    ("1 1001 1001 0 0", 0, "row"), ("64 8193 8193 0 0", 0, "row"), ("64 12288 12288 0 0", 0, "row"),
    ("64 12292 12292 0 0", 0, "top-k"), ("300 1001 1001 0 0", 0, "top-k"), ("64 4100 4100 0 0", 128, "row"),
    ("64 8193 8193 0 0", 128, "top-k"), ("64 4100 4100 0 0", 900, "top-k"),
    # large k
    ("64 1001 1001 112 1", 0, "top-k"), ("64 1001 1001 150 1", 0, "row"), ("64 12288 12288 150 1", 0, "top-k"),
    ("8 50257 50257 150 1", 0, "top-k"), ("8 151937 151937 496 1", 0, "row"), ("300 8193 8193 300 1", 0, "top-k"),
    ("300 8193 8193 496 1", 0, "row"), ("300 50257 50257 496 1", 0, "top-k"), ("64 8193 8193 300 1", 128, "row"),
    ("64 12288 12288 300 1", 128, "top-k"), ("600 1001 1001 496 1", 0, "top-k")])
def test_row_kernel_where_it_is_faster(host, call, history, kernel):
    """Calls whose rows are short or whose k is large run on the row kernel, as rows of odd length did before."""
    out = host(f"history {history} sample {call} 7")
    assert sum(f"{kernel} kernel" in line for line in out) == 1 and sum("kernel" in line for line in out) == 1, out
    assert out[-1] == "status 0"


def test_mapping_follows_the_resident_workgroups(host):
    """Rows eight apart only where eight rows' workgroups fit the device (64 places: one XCD of eight)."""
    for resident, rows, want in ((512, 64, 2), (512, 67, 1), (512, 300, 1), (64, 300, 1), (64, 40, 0), (64, 5, 0)):
        out = host(f"resident {resident} sample {rows} 151936 151936 0 1.0 7")
        assert f"mapping {want}" in out, (resident, rows, out)


BIG, ODD = "512 151936 151936 0 1.0", "512 151937 151937 0 1.0"


@pytest.mark.parametrize("call", [BIG, ODD])
def test_less_memory_takes_more_launches(host, call):
    """A workspace that cannot be had for all rows at once is asked for in half the rows, and again: 350 MB for the
    whole batch, 25 MB and several launches where that is all there is."""
    out = host(f"sample {call} 7")
    assert sum("fused kernel" in line for line in out) == 1 and out[-1] == "status 0", out
    out = host(f"memory 30000000 sample {call} 7 sample {call} 7")
    rows = [int(line.split()[2]) for line in out if line.startswith("fused kernel")]
    assert out.count("status 0") == 2 and sum(rows) == 2 * 512 and max(rows) <= 40, out
    assert not any("row kernel" in line for line in out)
    # an earlier call's smaller workspace, freed to make room for the larger, does not stop it either
    out = host(f"memory 30000000 sample 8 151936 151936 0 1.0 7 sample {call} 7 release 7")
    assert out.count("status 0") == 2 and sum(line.startswith("malloc ") and "failed" not in line for line in out) == \
        sum(line == "free block" for line in out), out


@pytest.mark.parametrize("call", [FULL, TOPK, ODD, "64 128257 128257 40 0.8"])
def test_no_memory_at_all_is_left_to_the_row_kernel(host, call):
    """... which needs none, for rows of every layout."""
    out = host(f"memory 0 sample {call} 7")
    assert sum("row kernel" in line for line in out) == 1 and out[-1] == "status 0", out


@pytest.mark.parametrize("call,small,kernel", [(FULL, "2 8192 8192 0 1.0", "fused"), (TOPK, "2 8192 8192 40 0.8", "top-k")])
def test_capture(host, call, small, kernel):
    """Nothing is allocated while a stream is captured: a call takes the workspace that an earlier one left, in as many
    launches as fit it, or else the row kernel."""
    out = host(f"capture 1 sample {call} 7")
    assert sum("row kernel" in line for line in out) == 1 and out[-1] == "status 0" and len(out) == 2, out
    out = host(f"sample {call} 7 capture 1 sample {call} 7")
    assert sum(f"{kernel} kernel, 64 rows" in line for line in out) == 2, out
    out = host(f"sample {small} 7 capture 1 sample {call} 7")
    assert not any("under capture" in line for line in out) and out[-1] == "status 0", out


@pytest.mark.parametrize("call,small", [(BIG, FULL), (ODD, "64 151937 151937 0 1.0"), ("512 128257 128257 112 1.0", TOPK)])
def test_captured_workspace_is_kept(host, call, small):
    """A graph holds the addresses of the workspace its calls were captured with: a later call that needs more leaves
    that one alone until the stream is released.  (One that no graph holds makes room.)"""
    out = host(f"sample {small} 7 capture 1 sample {small} 7 capture 0 sample {call} 7")
    assert sum(line.startswith("malloc ") for line in out) == 2 and not any("free" in line for line in out), out
    out = host(f"sample {small} 7 capture 1 sample {small} 7 capture 0 sample {call} 7 sample {call} 7 release 7")
    assert out[-3:] == ["free block", "free block", "release 0"], out
    out = host(f"sample {small} 7 sample {call} 7")
    assert sum("free block" in line for line in out) == 1, out


def test_greedy_slices(host):
    """Greedy slices of two batches only for long rows (at eight workgroups per CU)."""
    for call, want in (("64 128256 128256 0 0", 16), ("32 262144 262144 0 0", 32), ("300 16384 16384 0 0", 4),
                       ("128 32000 32000 0 0", 8)):
        assert f"slices {want}" in host(f"history 200 sample {call} 7"), call


def test_rows_in_halves_only_for_the_one_stream_of_large_grids(host):
    """Two grids with a row's workgroups in both halves can each hold half of every row: the mapping is left as soon as
    another stream has large grids, and comes back when that is released.  Small grids do not matter."""
    one, a, b = "sample 1 151936 151936 0 1.0", "sample 64 151936 151936 0 1.0 7", "sample 64 151936 151936 0 1.0 8"
    out = host(f"{one} 9 {a} {one} 9 {a} {b} {a} {b} release 7 {b}")
    assert [line for line in out if line.startswith("mapping")] == [f"mapping {m}" for m in (1, 2, 1, 2, 1, 1, 1, 2)], out
