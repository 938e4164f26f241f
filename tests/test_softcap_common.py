"""The branch-free soft-cap of the common range against the general restatement, on the host (the device runs both
over every float with cap 1 in test_gpu_sampler.py)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_softcap_common_range():
    exe = os.path.join(ROOT, "oracle", "_build", "softcap_common_check")
    src = os.path.join(ROOT, "tests", "native", "softcap_common_check.c")
    subprocess.run(["gcc", "-O2", "-mfma", "-ffp-contract=off", "-o", exe, src, "-lm"], check=True)
    caps = ["30", "50", "0.75", "1e4", "3.3333333", "1.0000001", "27.182818"]
    r = subprocess.run([exe, "499"] + caps, capture_output=True, text=True, timeout=300)
    rows = [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    assert len(rows) == len(caps) and all(n > 500000 and bad == 0 for n, bad, _, _ in rows), r.stdout
    # the wide form: all but NaN, quotients in [7.75, 16) and tiny ones
    assert all(wide > 1.2 * n and bad == 0 for n, _, wide, bad in rows), r.stdout


def test_softcap_caps_left_to_the_general_form():
    """Caps without a safe reciprocal: outside the exponent range, or a significand of all ones."""
    exe = os.path.join(ROOT, "oracle", "_build", "softcap_common_check")
    src = os.path.join(ROOT, "tests", "native", "softcap_common_check.c")
    subprocess.run(["gcc", "-O2", "-mfma", "-ffp-contract=off", "-o", exe, src, "-lm"], check=True)
    r = subprocess.run([exe, "99991", "1e-7", "1e13", "1.99999988", "inf"], capture_output=True, text=True, timeout=60)
    assert r.stdout.split() == ["0"] * 16, r.stdout
