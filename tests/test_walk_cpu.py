"""CPU check of the diagonal walk (latticeu1_amd/csrc/u1_walk.h) before it runs
on the GPU: the kernels' own address and order code, under random interleavings
that honour only the workgroup barrier, against two sequential phases with
brute-force coordinates (tests/cpu_checks/check_walk.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_walk_order_and_addresses(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = tmp_path / "check_walk"
    subprocess.run([hipcc, "-O2", "-std=c++17", os.path.join(HERE, "cpu_checks", "check_walk.cpp"), "-o", str(exe)],
                   check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "walk ok" in out.stdout
