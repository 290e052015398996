"""The kernels' FP32 operators act on constants as the FP64 ones do, and the
FP64 images are the operators (host build, no GPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC) or shutil.which("g++") is None, reason="needs hipcc")
def test_single_precision_operators_keep_constants(tmp_path):
    exe = tmp_path / "operators_check"
    cmd = [HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2", "-Wno-unused-function",
           "-I" + os.path.join(ROOT, "local-dg_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
           os.path.join(ROOT, "tests", "operators_check.cpp"), "-o", str(exe)]
    b = subprocess.run(cmd, capture_output=True, text=True)
    assert b.returncode == 0, b.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip().endswith("ok")
