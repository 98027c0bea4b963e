"""The staged host copies against a stand-in for the HIP calls, on the CPU
(tests/cpu/hostcopy_check.cpp): contexts of one device with uploads in flight,
in one thread and in several, failures in the middle of a copy, and the life of
the pinned slots."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


def test_host_copies_of_several_contexts(tmp_path):
    if not os.path.exists(HIPCC) and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    exe = str(tmp_path / "hostcopy_check")
    b = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O1", "-g", "-std=c++17",
                        "tests/cpu/hostcopy_check.cpp", "-o", exe, "-pthread"],
                       capture_output=True, text=True, cwd=ROOT, timeout=600)
    assert b.returncode == 0, b.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    assert "hostcopy_check: ok" in r.stdout
