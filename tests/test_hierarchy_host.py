"""Host-side checks of the Poisson V-cycle's set-up (tests/cpp/hierarchy_check.cpp, no GPU needed): the vertex
hierarchy and its packed matrices, the dense inverse, the line operators' eigenpairs."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ho-cxx_amd", "csrc")


def test_hierarchy(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    exe = tmp_path / "hierarchy_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, os.path.join(ROOT, "tests", "cpp", "hierarchy_check.cpp"),
                    os.path.join(CSRC, "hoc_host.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(out.stdout)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK"), out.stdout
