"""Device memory that a query call takes for its arrays, from the host code run on a stand-in for the
HIP runtime (tests/hip_stub.cpp): callers with device memory get temporaries only, host callers at
most 19 arrays of 4 bytes a ray where the staging is not bounded by 131,072 rays."""
import json

import pytest

from _hipstub import needs_stub, run

CODE = """
import json
n = %d
ctx = Context(0)
sc = scene_from_spec(ctx, scenes.cornell(1), commit=False)
if %d:
    sc.set_instances(0, np.eye(4, dtype=np.float32).reshape(1, 16))
sc.commit()
o, d = np.zeros((n, 3), np.float32), np.ones((n, 3), np.float32)
a = [np.zeros(n, np.float32) for _ in range(20)]
p = [x.ctypes.data for x in a]
rays = dict(zip(("org_x", "org_y", "org_z", "dir_x", "dir_y", "dir_z", "tnear", "tfar"), p))
hits = dict(zip(("t", "u", "v", "prim_id", "geom_id", "ng_x", "ng_y", "ng_z", "inst_id"), p[8:]))
recs = dict(zip(("distance", "prim_id", "geom_id", "material", "u", "v", "n_x", "n_y", "n_z", "p_x", "p_y", "p_z"), p[8:]))
sc.cast_rays(o[:1], d[:1])           # counters and the spill area
out = {}
for name, f in (("device", lambda: sc.cast_rays_device(rays, hits, n)),
                ("device records", lambda: sc.cast_ray_records_device(dict(rays, tfar=0), recs, n)),
                ("host any", lambda: sc.occluded(o, d)),
                ("host", lambda: sc.cast_rays(o, d, normals=True)),
                ("host records", lambda: sc.cast_ray_records(o, d, tnear=1e-3))):
    before = stub.stub_live()
    f()
    out[name] = stub.stub_live() - before
print(json.dumps(out))
"""


@needs_stub
@pytest.mark.parametrize("instanced", [0, 1])
@pytest.mark.parametrize("n", [200_000, 300_007])
def test_bytes_per_ray(tmp_path, n, instanced):
    # the stage is kept: what every call adds to the largest one before it
    grew = json.loads(run(CODE % (n, instanced), tmp_path))
    slack = 20 * 256 + 65536       # array alignment, the smallest block
    assert grew["device"] <= 4 * (1 + instanced) * n + slack, grew
    total, largest = grew["device"], 1 + instanced
    for name, arrays in (("device records", 5 + instanced), ("host any", 9), ("host", 18 + instanced),
                         ("host records", 19)):
        total, largest = total + grew[name], max(largest, arrays)
        assert total <= 4 * largest * n + slack, (name, total, grew)
