"""The append's fast e4m3 quantiser (fp8_code in csrc/kernels/append_body.h) equals
the reference's steps for every half value and every positive finite half scale,
checked by a host-only program built with hipcc (no GPU needed)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_fp8_fast_quantiser(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc is not available")
    exe = tmp_path / "fp8_code_check"
    src = os.path.join(HERE, "native", "fp8_code_check.cpp")
    r = subprocess.run([hipcc, "-O2", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-x", "hip", src, "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:]
