"""The MFMA decode uses no block-table entry past a row's own blocks (window_lane in
csrc/kernels/attention_body.h), checked by a host-only program built with hipcc (no
GPU needed)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_no_entry_past_the_row(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc is not available")
    exe = tmp_path / "block_window_check"
    src = os.path.join(HERE, "native", "block_window_check.cpp")
    r = subprocess.run([hipcc, "-O1", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-x", "hip", src, "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:]
