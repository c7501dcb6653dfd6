"""Work claiming of the query, engine and image kernels
(muon_amd/csrc/device/claim_plan.h): tests/cpu/claim_plan_check.cpp, built
with the host compiler against the header the kernels include, hands out
random item counts to random grids and checks that every item is taken once."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_item_claimed_once(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "claim_plan_check"
    src = os.path.join(ROOT, "tests", "cpu", "claim_plan_check.cpp")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-fsanitize=address,undefined",
                    "-I", os.path.join(ROOT, "muon_amd", "csrc", "device"), src, "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
