"""The exact traversal's quotients (muon_amd/csrc/device/exact_div.h) equal
IEEE division: tests/cpu/exact_div_check.cpp, built with the host compiler
against the header the kernels include, on every hard pair of significands."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_quotient_by_reciprocal(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "exact_div_check"
    src = os.path.join(ROOT, "tests", "cpu", "exact_div_check.cpp")
    cmd = ["g++", "-std=c++17", "-O2", "-Wall", "-ffp-contract=off", "-I",
           os.path.join(ROOT, "muon_amd", "csrc", "device"), src, "-o", str(exe)]
    with open("/proc/cpuinfo") as f:  # __builtin_fmaf: one instruction where there is one
        if " fma " in f.read():
            cmd.insert(1, "-mfma")
    subprocess.run(cmd, check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
