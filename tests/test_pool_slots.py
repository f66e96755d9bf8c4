"""The row-block kernels' pool slots (pool_slot and KeySlots in csrc/kernels/rows_body.h) do not
wrap at 2^31, checked by a host-only program
built with hipcc (no GPU needed)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_slots_past_32_bits(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc is not available")
    exe = tmp_path / "pool_slot_check"
    src = os.path.join(HERE, "native", "pool_slot_check.cpp")
    r = subprocess.run([hipcc, "-O1", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-x", "hip", src, "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:]
