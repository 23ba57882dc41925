"""Register counts of kernels whose speed hangs on the waves that share a SIMD
(512 vector registers: 128 a lane leave four waves, one more leaves three), read
from the assembly that hipcc writes for gfx950."""
import os
import re
import shutil
import subprocess

import pytest

from wgpufft_amd import build


def registers(source, tmp_path):
    """{kernel symbol: (vector registers, spilled ones)} of a HIP source."""
    hipcc = shutil.which(build.HIPCC)
    if hipcc is None:
        pytest.skip("hipcc is not installed")
    out = os.path.join(tmp_path, "kernels.s")
    flags = [f for f in build.COMMON if f != "-fPIC"]
    subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", os.path.join(build.CSRC, source), "-o", out], check=True,
                   capture_output=True)
    pattern = r"\.symbol: +(\S+)\.kd[\s\S]*?\.vgpr_count: +(\d+)\s+\.vgpr_spill_count: (\d+)"
    return {m[0]: (int(m[1]), int(m[2])) for m in re.findall(pattern, open(out).read())}


def test_register_bluestein_keeps_four_waves(tmp_path):
    """All points of a line and the loads in flight fit 128 registers up to 4096
    points (16 per thread)."""
    found = registers("kern_regconv.hip", tmp_path)
    for m in (64, 128, 256, 512, 1024, 2048, 4096):
        kernels = [v for k, v in found.items() if "RegBluesteinILi%dE" % m in k]
        assert kernels and all(v <= 128 and spilled == 0 for v, spilled in kernels), (m, kernels)
