"""Host checks of the launch limits and workspaces of key switches and rotations: which
batches a grouped launch holds, against block counts taken from the kernels' grids
(seal-cuda_amd/csrc/launch_limits.h), and the workspaces' layouts and sizes (workspaces.h:
regions apart, sizes that never shrink as the batch grows).  Host code only: no GPU needed."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "seal-cuda_amd", "csrc")


def run_check(tmp_path, name):
    exe = tmp_path / name
    src = os.path.join(HERE, "host", name + ".cpp")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", CSRC, src, "-o", str(exe)], check=True,
                   capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.startswith("ok ")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not on PATH")
def test_grouped_launches_are_taken_where_they_fit(tmp_path):
    run_check(tmp_path, "launch_limits_check")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not on PATH")
def test_workspaces_hold_smaller_batches(tmp_path):
    run_check(tmp_path, "workspaces_check")
