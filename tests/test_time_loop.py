"""The host side of trixi_hip_advance (csrc/time_loop.hpp), compiled for the host
from the header the library includes: steps and times of runs that end well and of
runs in which a launch or the wait fails at any step."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "trixicuda.jl_amd", "csrc")


def test_steps_and_times_after_success_and_failure(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "time_loop_check")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I", CSRC, os.path.join(HERE, "native", "time_loop_check.cpp"),
                    "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.split()[-1] == "ok", out.stdout
