"""A batch captures its graphs, and runs, on streams that no other call touches.

Calls beside it (reading a background renderer's image, cache calls, creating and resetting a
renderer) hold other locks than the batch: a launch of theirs on a stream in capture would go
into the batch's graph.  The library's host code runs here on a stand-in for the HIP runtime
that records the stream of every call."""
import json

from _hipstub import needs_stub, run

CODE = """
import json
ctx = Context(0)
sc = scene_from_spec(ctx, scenes.cornell(1))
def phase(name):
    stub.stub_phase(name.encode())
phase("renderer")
r = Renderer(ctx, sc, 64, 48, 2)
r.set_resolution(40, 30)
r.render(2)
r.reset()
phase("read")
r.raw(); r.current_progress(); r.current_normals(); r.current_stats()
phase("cache")
n = Nrc(ctx, max_batch=256)
q = np.zeros((64, 13), np.float32)
n.set_params(n.params()); n.infer(q); n.gradient(q, q[:, :3]); n.train_step(q, q[:, :3])
for graph in (True, False):
    for _ in range(2):
        phase("batch%d" % graph)
        render_batch(ctx, [dict(scene=sc, width=64, height=64, spp=4, max_bounces=2)], max_paths=4096, use_graph=graph)
        phase("rest")
        sc.cast_rays(np.zeros((5, 3), np.float32), np.ones((5, 3), np.float32))
        sc.commit()
print(json.dumps([l.split() for l in stub.stub_log().decode().splitlines()]))
"""


@needs_stub
def test_batch_streams_are_its_own(tmp_path):
    log = json.loads(run(CODE, tmp_path))
    null = "(nil)"
    captured = {s for _, f, s in log if f == "hipStreamBeginCapture"}
    assert captured
    assert all(p == "batch1" for p, f, _ in log if f == "hipStreamBeginCapture")
    batch = {s for p, _, s in log if p in ("batch0", "batch1") and s != null}
    others = {s for p, _, s in log if p not in ("batch0", "batch1") and s != null}
    assert captured <= batch and not batch & others, (captured, batch, others)
    # two sets, kept between the calls
    assert len(batch) == 2
    assert sum(f == "hipStreamCreateWithFlags" for p, f, _ in log if p.startswith("batch")) == 2
    # nothing but the recorded kernels reaches a stream in capture
    inside = False
    for p, f, s in log:
        if f == "hipStreamBeginCapture":
            inside = True
        elif f == "hipStreamEndCapture":
            inside = False
        elif inside:
            assert f == "hipLaunchKernel", f
