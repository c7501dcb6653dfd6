"""Host-side checks of the headers that the kernels and their launches share:
each program in tests/cpu named here is built with the host C++ compiler
against muon_amd/csrc/device, under the sanitizers, and prints "ok"."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("name", ["poll_plan_check", "path_capacity_check",
                                  "query_parts_check"])
def test_cpu_check(name, tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / name
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-fsanitize=address,undefined",
                    "-I", os.path.join(ROOT, "muon_amd", "csrc", "device"),
                    os.path.join(ROOT, "tests", "cpu", name + ".cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
