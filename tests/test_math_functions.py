"""sincos_cr and pow5_cr (crt_math.h) against the host's FP64 functions rounded to FP32.

Both sides are within about one FP64 unit of the exact value, so they round to different FP32
numbers only where the exact value lies within 2^-53 relative of a rounding boundary, which
are 2^-24 apart: about one result in 2^28.  Over 2^25 sines and cosines that is an eighth of a
result, over 2^24 fifth powers (three roundings) a quarter; four of each are allowed, and no
difference may exceed one FP32 unit.  The sun's threshold has to agree with the angle it
stands for at every cosine tried."""
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


@pytest.mark.skipif(shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists(),
                    reason="hipcc not available")
def test_fp64_rounded_functions(tmp_path):
    exe = tmp_path / "probe"
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    subprocess.run([hipcc, "-O2", "-std=c++17", "--offload-arch=gfx950", "-ffp-contract=off",
                    f"-I{HERE.parent / 'crender_amd' / 'csrc'}", str(HERE / "math_probe.cpp"), "-o", str(exe)], check=True,
                   capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()
    trig, fifth, worst, sides = (int(v) for v in out)
    assert trig <= 4 and fifth <= 4 and worst <= 1 and sides == 0, out
