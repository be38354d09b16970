"""The deepest stack of an admitted scene (264 entries) fits wherever the rules send its rays: a
lane's LDS stack and spill area, or the LDS of the eight lanes of a ray, 64, 128 or 256 entries."""
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not available")
def test_stack_rules(tmp_path):
    exe = tmp_path / "probe"
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-arch=gfx950", f"-I{HERE.parent / 'crender_amd' / 'csrc'}",
                    f"-I{HERE.parent / 'include'}", str(HERE / "stack_probe.cpp"), "-o", str(exe)], check=True,
                   capture_output=True)
    bad, group = (int(v) for v in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split())
    assert bad == 0
    assert group == 65 + 129 + 257   # needs 0 .. 64, 128 and 256; 257 to 264 stay with a lane per ray
