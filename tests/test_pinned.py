"""The rule for host memory that the server reads in place (katric_amd/csrc/kt_pinned.h)."""
import os
import subprocess

from tests.conftest import ROOT


def test_only_ranges_inside_one_page_locked_allocation(tmp_path):
    exe = tmp_path / "test_pinned"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", os.path.join(ROOT, "tests", "cpp", "test_pinned.cpp"),
                    "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0 and "ALL OK" in res.stdout, res.stdout + res.stderr
