"""CPU check of the control words of one-launch sweeps
(latticeu1_amd/csrc/u1_die_sync.h): the kernel's own code, with accesses that
complete late and in any order it does not rule out, several launches in a row
(tests/cpu_checks/check_die_sync.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_control_words(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = tmp_path / "check_die_sync"
    subprocess.run([hipcc, "-O2", "-std=c++17", os.path.join(HERE, "cpu_checks", "check_die_sync.cpp"), "-o", str(exe)],
                   check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "die sync ok" in out.stdout
