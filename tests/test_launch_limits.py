"""Host checks of the key switch's launch limits (seal-cuda_amd/csrc/launch_limits.h): which
batches a grouped launch holds, against block counts taken from the kernels' grids.  Host
code only: no GPU needed."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "seal-cuda_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not on PATH")
def test_grouped_launches_are_taken_where_they_fit(tmp_path):
    exe = tmp_path / "launch_limits_check"
    src = os.path.join(HERE, "host", "launch_limits_check.cpp")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", CSRC, src, "-o", str(exe)], check=True,
                   capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.startswith("ok ")
