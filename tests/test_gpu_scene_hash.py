"""The scene hash of a checkpoint, computed on the device in chunks, against the byte by byte
FNV-1a chain over the same arrays: per model its corners, local material indices and materials,
then the sky, then the instances.  Sizes around the chunks (1024 bytes), the spans of 128 chunks
and the rounds of 65,536 chunks (64 MB)."""
import ctypes as C
import shutil
import struct
import subprocess

import numpy as np
import pytest

from crender_amd import Context, Renderer, Scene, scenes
from crender_amd.render import _material

pytestmark = pytest.mark.gpu

SRC = """#include <stdint.h>
#include <stddef.h>
uint64_t fnv(uint64_t h, const uint8_t *p, size_t n)
{ for (size_t i = 0; i < n; ++i) h = (h ^ p[i]) * 1099511628211ull; return h; }
"""


@pytest.fixture(scope="module")
def fnv(tmp_path_factory):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    d = tmp_path_factory.mktemp("fnv")
    (d / "fnv.c").write_text(SRC)
    subprocess.run([cc, "-O2", "-shared", "-fPIC", str(d / "fnv.c"), "-o", str(d / "fnv.so")], check=True)
    f = C.CDLL(str(d / "fnv.so")).fnv
    f.restype, f.argtypes = C.c_uint64, [C.c_uint64, C.c_char_p, C.c_size_t]

    def run(parts):
        h = 1469598103934665603
        for b in parts:
            h = f(h, b, len(b))
        return h

    return run


def _soup(n, seed):
    rng = np.random.default_rng(seed)
    v = rng.random((3 * n, 3), dtype=np.float32)
    mats = [scenes.MaterialSpec(colour=(0.1 * k, 0.5, 0.5, 1.0)) for k in range(3)]
    return scenes.SceneSpec(name="s", vertices=v, vertex_indices=np.arange(3 * n, dtype=np.uint32),
                            material_indices=rng.integers(0, 3, n).astype(np.uint32), materials=mats,
                            camera=scenes.camera_dict((0.5, 0.5, -1.0)))


@pytest.mark.parametrize("sizes,sky,instances", [([1], None, 0), ([28], (1, 1), 0), ([29], (3, 2), 0), ([256], None, 3),
                                                 ([3640, 1, 3641], (16, 8), 0), ([7000, 512], None, 2),
                                                 ([1_900_000], (64, 32), 0)])
def test_hash_equals_byte_chain(fnv, sizes, sky, instances):
    ctx = Context(0)
    sc = Scene(ctx)
    parts, inst_parts = [], []
    for k, n in enumerate(sizes):
        spec = _soup(n, 31 + k)
        sc.add_model(spec)
        parts += [spec.corners().tobytes(), spec.material_indices.tobytes(),
                  b"".join(bytes(_material(m)) for m in spec.materials)]
        m = np.eye(4, dtype=np.float32).reshape(1, 16)
        if instances:
            m = np.repeat(m, instances, 0)
            m[:, 12] = np.arange(instances) * 2.0
            sc.set_instances(k, m)
        inst_parts.append(m.tobytes())
    if sky:
        img = np.random.default_rng(5).random((sky[1], sky[0], 4), dtype=np.float32)
        sc.set_skybox(img)
        parts.append(img.tobytes())
    if instances:
        parts += inst_parts
    sc.set_camera(spec.camera)
    for _ in range(2):   # a second commit hashes the same arrays again
        sc.commit()
        r = Renderer(ctx, sc, 4, 4, 1)
        got = struct.unpack_from("<Q", r.checkpoint(), 56)[0]
        r.close()
        assert got == fnv(parts)
    sc.close()
    ctx.close()
