"""A plan for combined images where the system has no threads left: the fit runs
on the caller's thread, and no exception leaves the library."""
import os
import shutil
import subprocess

import pytest

from tests.test_kernel_cpu_build import ROOT


def test_fit_without_threads(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "lowrank_threads_cpu")
    cmd = [gxx, "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "pytomography_amd", "csrc"),
           os.path.join(ROOT, "tests", "cpu_build", "lowrank_threads_cpu.cpp"), "-ldl", "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "same 1", (r.returncode, r.stdout, r.stderr)
