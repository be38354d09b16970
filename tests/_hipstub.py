"""Runs host code of the library in a process of its own against tests/hip_stub.cpp."""
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
HIP_INCLUDE = Path("/opt/rocm/include")

needs_stub = pytest.mark.skipif(shutil.which("g++") is None or not (HIP_INCLUDE / "hip" / "hip_runtime_api.h").exists(),
                                reason="g++ or the HIP headers are not available")

PRELUDE = """
import ctypes as C, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)   # ahead of libcrt.so and the runtime it links
stub.stub_log.restype = C.c_char_p
stub.stub_phase.argtypes = [C.c_char_p]
stub.stub_fail.argtypes = [C.c_long]
stub.stub_handles.restype = C.c_long
stub.stub_live.restype = C.c_size_t
sys.path[:0] = [%r, %r]
import numpy as np
from crender_amd import Context, CrtError, Nrc, Renderer, render_batch, scene_from_spec, scenes
"""


def run(code: str, tmp: Path) -> str:
    """Output of `code` (after PRELUDE), run by a Python of its own."""
    lib = tmp / "hip_stub.so"
    subprocess.run(["g++", "-O1", "-std=gnu++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", f"-I{HIP_INCLUDE}",
                    str(HERE / "hip_stub.cpp"), "-o", str(lib)], check=True, capture_output=True)
    p = subprocess.run([sys.executable, "-c", PRELUDE % (str(HERE.parent), str(HERE)) + code, str(lib)],
                       capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stderr[-3000:]
    return p.stdout
