"""The intersection's bin rule (katric_amd/csrc/kt_bins.h), enumerated on the host."""
import os
import subprocess

from tests.conftest import ROOT


def test_every_tail_gets_a_bucket_of_its_class(tmp_path):
    exe = tmp_path / "test_bins"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", os.path.join(ROOT, "tests", "cpp", "test_bins.cpp"),
                    "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0 and "ALL OK" in res.stdout, res.stdout + res.stderr
