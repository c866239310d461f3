"""The small one-launch solve reads no slot outside a row's own slice, with whole
slices of rows without entries too (sell_slot, elfel.jl_amd/csrc/nine.h).
tests/small_slots_check.cpp is a host-only program (no device calls: runs
without a GPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC) and shutil.which("hipcc") is None, reason="hipcc not installed")
def test_slots_are_the_rows_own(tmp_path):
    hipcc = HIPCC if os.path.exists(HIPCC) else shutil.which("hipcc")
    exe = tmp_path / "small_slots_check"
    subprocess.run([hipcc, "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "elfel.jl_amd", "csrc"),
                    os.path.join(ROOT, "tests", "small_slots_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout + r.stderr
