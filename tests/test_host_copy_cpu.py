"""Host code against a stand-in for the HIP calls, on the CPU: the staged copies
(tests/cpu/hostcopy_check.cpp), with contexts of one device and uploads in flight,
in one thread and in several, failures in the middle of a copy, and the life of
the pinned slots; and buffers that cannot grow (tests/cpu/alloc_check.cpp)."""
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


def test_buffers_after_a_failed_allocation(tmp_path):
    """The context's growing buffers against a stand-in for the allocation calls
    (tests/cpu/alloc_check.cpp); kernels are not linked, none is launched."""
    if not os.path.exists(HIPCC) and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    exe = str(tmp_path / "alloc_check")
    b = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O1", "-g", "-std=c++17",
                        "tests/cpu/alloc_check.cpp", "-o", exe,
                        "-Wl,--unresolved-symbols=ignore-all"],
                       capture_output=True, text=True, cwd=ROOT, timeout=600)
    assert b.returncode == 0, b.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr[-3000:]
    assert "alloc_check: ok" in r.stdout
