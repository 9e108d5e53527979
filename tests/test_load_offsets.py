"""The activation loads of the kernels stay inside x (CPU only): tests/load_offsets.cpp walks the buffer
offsets that csrc/qmm4_offsets.h gives them, over rows around each row block's size."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_rows_past_the_end_are_never_read(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ is not available")
    exe = str(tmp_path / "load_offsets")
    cmd = [cxx, "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
           "-I", os.path.join(ROOT, "mlx-tree-spec_amd", "csrc"), os.path.join(ROOT, "tests", "load_offsets.cpp"),
           "-o", exe]
    build = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr[-4000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stdout[-4000:]
    assert "violations: 0" in run.stdout
