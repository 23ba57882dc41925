"""The host planner of the register-stage kernels (mix_plan.cpp), compiled as it
is with tests/mix_plan/driver.cpp: over every smooth length up to 2^15, f32 and
f64, contiguous and strided, standalone and batched, lines, half-length real
lines and convolutions, a tile of one buffer fits one round, no stage leaves the
LDS pitch, every (radix, unroll) pair is a compiled one and every division is in
its range (a violation would be a race in LDS or a skipped stage), a line run at
a tile's addresses is a DFT, and the schedule search finds what a search of every
order finds."""
import os
import shutil
import subprocess

import pytest

from wgpufft_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_tiles_and_schedules(tmp_path):
    hipcc = shutil.which(build.HIPCC)
    if hipcc is None:
        pytest.skip("hipcc is not installed")
    exe = os.path.join(tmp_path, "mix_plan_driver")
    subprocess.run([hipcc, "-O2", "-std=c++17", "-x", "hip", "--offload-host-only", "-Wno-unused-result", "-I", build.CSRC,
                    "-I", os.path.join(build.HERE, "..", "include"), os.path.join(HERE, "mix_plan", "driver.cpp"), "-o", exe],
                   check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    assert "checked 1201 schedules" in r.stdout, r.stdout
