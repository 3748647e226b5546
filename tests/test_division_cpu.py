"""Quotients by reciprocal and two correction steps are the divisions'
(affine_quantize8 and unit_run), on the CPU's fused multiply-add."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_corrected_quotients(tmp_path):
    exe = str(tmp_path / "division_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wall", "-Wno-parentheses",
                    os.path.join(HERE, "native", "division_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
