"""A commit that fails at any of its HIP calls returns an error, leaves a scene that can be committed
again or closed, and no device memory, event or
stream behind.  The library's host code runs on a stand-in for
the HIP runtime (tests/hip_stub.cpp) whose k-th call fails."""
import json

import pytest

from _hipstub import needs_stub, run

CODE = """
import json
spec = scenes.cutout(3) if %d else scenes.cornell(1)
def scene(ctx):
    sc = scene_from_spec(ctx, spec, commit=False)
    if %d:
        sc.set_instances(0, np.eye(4, dtype=np.float32).reshape(1, 16))
    return sc
ctx = Context(0)
scene(ctx).commit()                  # the builder's scratch is kept until the process ends
ctx.close()
base = stub.stub_live(), stub.stub_handles()
failed, leaks, again = 0, [], 0
for k in range(400):
    ctx = Context(0)
    sc = scene(ctx)
    stub.stub_clear()
    stub.stub_fail(k)
    try:
        sc.commit()
        ok = True
    except CrtError:
        ok = False
    stub.stub_fail(-1)
    reached = stub.stub_reached(k)
    if not ok:
        failed += 1
        if k %% 7 == 0:
            sc.commit()
            again += 1
    ctx.close()
    now = stub.stub_live(), stub.stub_handles()
    if now != base:
        leaks.append((k, now[0] - base[0], now[1] - base[1]))
        base = now
    if not reached:
        break
print(json.dumps(dict(failed=failed, leaks=leaks, again=again, calls=k)))
"""


@needs_stub
@pytest.mark.parametrize("textured,instanced", [(0, 0), (1, 0), (0, 1)])
def test_nothing_is_left_behind(tmp_path, textured, instanced):
    r = json.loads(run(CODE % (textured, instanced), tmp_path))
    assert r["failed"] > 20 and r["calls"] < 399, r
    assert r["leaks"] == []
