"""The arrival counter of the device reductions (csrc/arrival.hpp), compiled for
the host from the header the kernels include: after any order of arrival of
launches that overlap, the counter is at zero and later launches find their last
block."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "trixicuda.jl_amd", "csrc")


def test_counter_recovers_from_every_overlap(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "arrival_check")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I", CSRC, os.path.join(HERE, "native", "arrival_check.cpp"),
                    "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.split()[-1] == "ok", out.stdout
