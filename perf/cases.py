"""Timed workloads of the path tracer, each one pass through the library's public entry points.

A case is a dict of plain values with a ``kind``:

  query     a batch of rays against a committed scene (``Scene.cast_rays_device``,
            ``cast_rays``, ``cast_ray_records``, ``occluded``)
  render    a fresh accumulation of ``spp`` passes by a ``Renderer``
  batch     many scenes rendered together (``render_batch``)
  infer     radiance-cache predictions of a frame's queries (``crt_nrc_infer``)
  gradient  forward and backward of the radiance cache's network (``crt_nrc_gradient``)
  finish    a frame's denoising and the post-processing of a displayed image
            (``crt_denoise``, ``crt_post_process``)
  load      a model handed to a new scene, its commit, and the first rays cast into it

``listed()`` names the fixed cases, ``draw(rng)`` gives further ones of the same ranges,
``prepare`` / ``run`` build a state and take one pass, ``work`` counts the bytes and
operations a pass cannot do without, and ``exact`` restates the numeric ones in FP64.
"""
import ctypes as C
import math

import numpy as np
import torch

from crender_amd import (Context, Nrc, Renderer, Scene, _abi as A, denoise, post_process, render_batch,
                         scene_from_spec, scenes)

DEV = "cuda"
F32, F64 = torch.float32, torch.float64
RAY_KEYS = ("org_x", "org_y", "org_z", "dir_x", "dir_y", "dir_z", "tnear", "tfar")
HIT_KEYS = ("t", "u", "v", "prim_id", "geom_id", "ng_x", "ng_y", "ng_z", "inst_id")
INT_KEYS = ("prim_id", "geom_id", "inst_id", "material")
LAYERS = ((96, 64), (64, 64), (64, 64), (64, 64), (64, 64), (64, 32))   # the cache's MLP


def listed():
    return [
        # mouse picking and gameplay probes: a handful of rays, all latency
        {"name": "pick-rays-96", "kind": "query", "call": "closest", "memory": "device", "rays": "diffuse",
         "n": 96, "tris": 100_000, "instances": 1},
        # primary visibility of a 1080p frame on the million-triangle soup, rays resident on the GPU
        {"name": "camera-rays-1080p", "kind": "query", "call": "closest", "memory": "device", "rays": "camera",
         "n": 1920 * 1080, "tris": 1_000_000, "instances": 1},
        # a host tool asking for full intersection records on a scene of placed instances
        {"name": "records-host-instances", "kind": "query", "call": "records", "memory": "host", "rays": "diffuse",
         "n": 65_537, "tris": 5_000, "instances": 16},
        # the Cornell box at its own settings: small launches, many bounces, image read back
        {"name": "render-cornell-256", "kind": "render", "scene": "cornell", "tris": 36, "width": 256, "height": 256,
         "spp": 16, "bounces": 8, "rr": 3, "mode": 0},
        # the headline workload: 1M-triangle soup, 1080p, primary plus three diffuse bounces
        {"name": "render-soup-1080p", "kind": "render", "scene": "soup", "tris": 1_000_000, "width": 1920,
         "height": 1080, "spp": 8, "bounces": 4, "rr": 0, "mode": 0},
        # terrain with diffuse, metal and glass spheres under sun and sky, physically based, depth 8
        {"name": "render-terrain-1080p", "kind": "render", "scene": "terrain", "tris": 1_000_000, "width": 1920,
         "height": 1080, "spp": 12, "bounces": 8, "rr": 3, "mode": 1},
        # textures, alpha cut-outs and an image sky with sun shadows: the interactive preview
        {"name": "render-textured-640", "kind": "render", "scene": "cutout", "tris": 44, "width": 640, "height": 360,
         "spp": 4, "bounces": 6, "rr": 3, "mode": 0},
        # a thumbnail service: scenes of different sizes and resolutions in one batch
        {"name": "batch-8-scenes", "kind": "batch", "jobs": 8, "tris": 60_000, "edge": 512, "spp": 8, "bounces": 4},
        # one cache query per pixel of a 1080p frame
        {"name": "cache-infer-1080p", "kind": "infer", "n": 1920 * 1080},
        # one training batch of the cache, forward and backward
        {"name": "cache-gradient-16k", "kind": "gradient", "n": 16_384},
        # denoise and tone-map a 1080p frame that stays on the GPU
        {"name": "finish-frame-1080p", "kind": "finish", "memory": "device", "width": 1920, "height": 1080,
         "levels": 5, "tonemap": 3, "gray": 0, "full": 0},
        # bring a model in: copy, build, first rays
        {"name": "load-model-400k", "kind": "load", "tris": 400_003, "n": 1_024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["query", "query", "query", "render", "render", "batch", "infer", "gradient", "finish", "load"])
    if kind == "query":
        call = rng.choice(["closest", "closest", "records", "occluded"])
        memory = "host" if call == "occluded" else rng.choice(["device", "host"])
        inst = rng.choice([1, 1, 1, rng.randint(2, 16)])
        return {"kind": kind, "call": call, "memory": memory, "rays": rng.choice(["camera", "diffuse"]),
                "n": _log(rng, 1, 2_000_000 if memory == "device" else 250_000),
                "tris": _log(rng, 500, 1_000_000 if inst == 1 else 50_000), "instances": inst}
    if kind == "render":
        scene = rng.choice(["cornell", "soup", "terrain", "cutout"])
        w, h = _log(rng, 96, 1920), _log(rng, 64, 1080)
        return {"kind": kind, "scene": scene, "tris": _log(rng, 2_000, 1_000_000), "width": w, "height": h,
                "spp": rng.randint(1, 8 if scene != "cutout" else 4), "bounces": rng.randint(2, 6),
                "rr": rng.choice([0, 3]), "mode": rng.choice([0, 1])}
    if kind == "batch":
        return {"kind": kind, "jobs": rng.randint(2, 8), "tris": _log(rng, 2_000, 60_000),
                "edge": rng.randint(96, 512), "spp": rng.randint(1, 8), "bounces": rng.randint(2, 4)}
    if kind == "infer":
        return {"kind": kind, "n": _log(rng, 1, 1920 * 1080)}
    if kind == "gradient":
        return {"kind": kind, "n": _log(rng, 64, 65_536)}
    if kind == "finish":
        return {"kind": kind, "memory": rng.choice(["device", "host"]), "width": _log(rng, 64, 1920),
                "height": _log(rng, 48, 1080), "levels": rng.randint(1, 5), "tonemap": rng.randint(0, 3),
                "gray": rng.choice([0, 0, 1]), "full": rng.choice([0, 1])}
    return {"kind": kind, "tris": _log(rng, 1_000, 400_000), "n": _log(rng, 64, 4_096)}


# ---- inputs, made from the seed alone ------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(0x5EED + 7919 * seed)


def _rand(g, *shape):
    return torch.rand(shape, generator=g, device=DEV, dtype=F32)


def _unit(g, n):
    z = 2.0 * _rand(g, n) - 1.0
    ph = 2.0 * math.pi * _rand(g, n)
    r = torch.sqrt(torch.clamp(1.0 - z * z, min=0.0))
    return torch.stack([r * torch.cos(ph), r * torch.sin(ph), z], 1)


def _soup_vertices(g, n):
    """(3n, 3) corners of n random triangles in the unit cube, their size falling with n."""
    sigma = 0.005 * (1e6 / n) ** (1.0 / 3.0)
    cen = _rand(g, n, 1, 3)
    off = torch.randn((n, 3, 3), generator=g, device=DEV, dtype=F32) * sigma
    return (cen + off).reshape(-1, 3)


def _soup_spec(verts, name="soup"):
    v = verts.cpu().numpy()
    n = v.shape[0] // 3
    return scenes.SceneSpec(name=name, vertices=v, vertex_indices=np.arange(3 * n, dtype=np.uint32),
                            material_indices=np.zeros(n, np.uint32),
                            materials=[scenes.MaterialSpec(colour=(0.8, 0.8, 0.8, 1.0))], sky=scenes.constant_sky(1.0),
                            sun_enabled=False, camera=scenes.camera_dict((0.5, 0.5, -1.0), fov=60.0))


def _transforms(g, k):
    """k column-major object-to-world matrices: rotation, uniform scale, placement on a jittered grid."""
    out = np.zeros((k, 4, 4), np.float64)
    u = _rand(g, k, 8).cpu().numpy().astype(np.float64)
    side = max(1, math.ceil(k ** (1.0 / 3.0)))
    for i in range(k):
        axis = u[i, :3] - 0.5
        axis /= max(np.linalg.norm(axis), 1e-6)
        a, s = 2.0 * math.pi * u[i, 3], 0.5 + 0.4 * u[i, 4]
        kx = np.array([[0, -axis[2], axis[1]], [axis[2], 0, -axis[0]], [-axis[1], axis[0], 0]])
        rot = np.eye(3) + math.sin(a) * kx + (1.0 - math.cos(a)) * (kx @ kx)
        m = np.eye(4)
        m[:3, :3] = s * rot
        cell = np.array([i % side, (i // side) % side, i // (side * side)], np.float64)
        m[:3, 3] = cell + 0.2 * u[i, 5:8]
        out[i] = m.T
    return out.reshape(k, 16).astype(np.float32)


def _rays(g, case):
    """(8, n) rays: org, dir, tnear, tfar."""
    n = case["n"]
    side = max(1.0, float(math.ceil(case.get("instances", 1) ** (1.0 / 3.0))))
    if case.get("rays") == "camera":
        w = max(1, int(math.ceil(math.sqrt(n * 16.0 / 9.0))))
        h = (n + w - 1) // w
        i = torch.arange(n, device=DEV)
        x = (i % w).to(F32) + _rand(g, n)
        y = (i // w).to(F32) + _rand(g, n)
        d = torch.stack([(2.0 * x / w - 1.0) * (w / h), 2.0 * y / h - 1.0, torch.full_like(x, 1.7320508)], 1)
        d = d / d.norm(dim=1, keepdim=True)
        o = torch.tensor([0.5 * side, 0.5 * side, -1.0 * side], device=DEV, dtype=F32).expand(n, 3)
    else:
        o = _rand(g, n, 3) * side
        d = _unit(g, n)
    r = torch.empty((8, n), device=DEV, dtype=F32)
    r[0:3] = o.T
    r[3:6] = d.T
    r[6] = 1e-5
    r[7] = math.inf if case.get("call") != "occluded" else 0.5 * side   # sun or lamp at a distance
    return r.contiguous()


def _query_inputs(case, seed):
    g = _gen(seed)
    verts = _soup_vertices(g, case["tris"])
    inst = _transforms(g, case["instances"]) if case["instances"] > 1 else None
    return verts, inst, _rays(g, case)


def _net(seed):
    """Kaiming-uniform weights of the cache's network, (K, N) per layer, zero padding."""
    g = _gen(seed)
    ws = []
    for i, (k, n) in enumerate(LAYERS):
        fan = 83 if i == 0 else k
        w = (2.0 * _rand(g, k, n) - 1.0) * math.sqrt((3.0 if i == 5 else 6.0) / fan)
        if i == 0:
            w[83:] = 0.0
        if i == 5:
            w[:, 3:] = 0.0
        ws.append(w)
    return ws, g


def _cache_queries(g, n):
    """(n, 13): position in the scene box, direction, normal, albedo, roughness."""
    rough = torch.where(_rand(g, n, 1) < 0.7, torch.ones((n, 1), device=DEV), _rand(g, n, 1) * 0.5)
    return torch.cat([_rand(g, n, 3), _unit(g, n), _unit(g, n), 0.2 + 0.7 * _rand(g, n, 3), rough], 1).contiguous()


def _frame(g, h, w):
    """(H, W, 4) colour, normal and albedo images of a noisy frame with object edges."""
    def patches(cells, lo, hi):
        low = lo + (hi - lo) * _rand(g, 1, 3, cells, cells)
        img = torch.nn.functional.interpolate(low, size=(h, w), mode="nearest")[0].permute(1, 2, 0)
        return img.contiguous()

    alb = patches(24, 0.1, 0.9)
    nrm = patches(16, 0.0, 1.0)
    noise = 0.5 + _rand(g, h, w, 3)
    col = alb * noise + (_rand(g, h, w, 1) < 0.002).to(F32) * 2.0   # fireflies
    one = torch.ones((h, w, 1), device=DEV, dtype=F32)
    return [torch.cat([x, one], 2).contiguous() for x in (col, nrm, alb)]


def _finish_inputs(case, seed):
    g = _gen(seed)
    h, w = case["height"], case["width"]
    col, nrm, alb = _frame(g, h, w)
    return col, nrm, alb, _frame(g, h, w)[0]   # the last: the image being displayed


def _render_spec(case, seed):
    g = _gen(seed)
    if case["scene"] == "cornell":
        return scenes.cornell(seed)
    if case["scene"] == "cutout":
        return scenes.cutout(seed, mode=case["mode"])
    if case["scene"] == "soup":
        return _soup_spec(_soup_vertices(g, case["tris"]))
    spheres = max(1, case["tris"] // 1100)
    grid = max(4, int(math.sqrt(max(case["tris"] - 320 * spheres, 32) / 2)) + 1)
    return scenes.terrain(grid=grid, spheres=spheres, seed=seed)


# ---- prepare ------------------------------------------------------------------------------

class _DeviceView:
    """Lets torch read a device buffer of a renderer in place; the tensor made from it holds
    the view, and the view the renderer, whose buffer it is."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f4", "version": 3,
                                         "strides": None}


def _device_buffer(r, which, shape):
    p = C.c_void_p()
    A.check(A.lib().crt_renderer_device_buffer(r._h, A.BUFFER[which], C.byref(p)))
    return torch.as_tensor(_DeviceView(r, p.value, shape), device=DEV)


def _query_scene(ctx, verts, inst):
    sc = scene_from_spec(ctx, _soup_spec(verts), commit=False)
    if inst is not None:
        sc.set_instances(0, inst)
    sc.commit()
    return sc


def prepare(case, seed):
    kind = case["kind"]
    ctx = Context(0)
    st = {"case": case, "ctx": ctx}
    if kind == "query":
        verts, inst, rays = _query_inputs(case, seed)
        st["scene"] = _query_scene(ctx, verts, inst)
        n = case["n"]
        if case["memory"] == "host":
            r = rays.cpu().numpy()
            st["org"], st["dir"] = np.ascontiguousarray(r[0:3].T), np.ascontiguousarray(r[3:6].T)
            st["tnear"], st["tfar"] = float(r[6, 0]), float(r[7, 0])
        else:
            st["rays"] = rays
            st["ray_ptrs"] = {k: rays[i].data_ptr() for i, k in enumerate(RAY_KEYS)}
            keys = HIT_KEYS if case["call"] == "closest" else A.RECORD_FIELDS
            st["out"] = {k: torch.empty(n, device=DEV, dtype=torch.int32 if k in INT_KEYS else F32) for k in keys}
            st["out_ptrs"] = {k: t.data_ptr() for k, t in st["out"].items()}
    elif kind == "render":
        spec = _render_spec(case, seed)
        st["scene"] = scene_from_spec(ctx, spec)
        r = Renderer(ctx, st["scene"], case["width"], case["height"], case["bounces"])
        r.set_resolution(case["width"], case["height"])
        r.set_options(mode=case["mode"], rr_start=case["rr"], seed=seed)
        st["renderer"] = r
    elif kind == "batch":
        st["jobs"], st["scenes"] = [], []
        for k in range(case["jobs"]):
            part = 1.0 - 0.6 * k / case["jobs"]   # the later jobs are smaller
            tris, edge = max(500, int(case["tris"] * part)), max(32, int(case["edge"] * part))
            spec = _render_spec({"scene": "soup" if k % 2 == 0 else "terrain", "tris": tris}, seed * 64 + k)
            st["scenes"].append(scene_from_spec(ctx, spec))
            st["jobs"].append({"scene": st["scenes"][-1], "width": edge, "height": edge - k, "mode": k % 2,
                               "spp": max(1, int(case["spp"] * part)),
                               "max_bounces": case["bounces"], "rr_start": 3, "seed": seed + k})
    elif kind in ("infer", "gradient"):
        ws, g = _net(seed)
        n = case["n"]
        st["nrc"] = Nrc(ctx, max_batch=65_536, seed=1)
        st["nrc"].set_params(torch.cat([w.reshape(-1) for w in ws]).cpu().numpy())
        st["queries"] = _cache_queries(g, n)
        if kind == "infer":
            st["out"] = torch.empty((n, 3), device=DEV, dtype=F32)
        else:
            st["targets"] = _cache_targets(g, n)
            st["grad"] = np.empty(st["nrc"].n_params, np.float32)
    elif kind == "finish":
        imgs = _finish_inputs(case, seed)
        if case["memory"] == "host":
            st["images"] = [x.cpu().numpy() for x in imgs]
        else:
            st["images"] = imgs
            st["denoised"], st["shown"] = torch.empty_like(imgs[0]), torch.empty_like(imgs[3])
    else:
        verts, rays = _load_inputs(case, seed)
        st["spec"] = _soup_spec(verts, "model")
        r = rays.cpu().numpy()
        st["org"], st["dir"] = np.ascontiguousarray(r[0:3].T), np.ascontiguousarray(r[3:6].T)
    torch.cuda.synchronize()
    return st


def _cache_targets(g, n):
    return (_rand(g, n, 3) * torch.exp(0.8 * torch.randn((n, 1), generator=g, device=DEV, dtype=F32))).contiguous()


def _load_inputs(case, seed):
    g = _gen(seed)
    verts = _soup_vertices(g, case["tris"])
    return verts, _rays(g, {"n": case["n"], "rays": "diffuse"})


# ---- run ----------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    return globals()["_run_" + case["kind"]](case, state)


def _run_query(case, st):
    sc = st["scene"]
    if case["memory"] == "device":
        if case["call"] == "closest":
            sc.cast_rays_device(st["ray_ptrs"], st["out_ptrs"], case["n"])
        else:
            sc.cast_ray_records_device(st["ray_ptrs"], st["out_ptrs"], case["n"])
        return st["out"]
    if case["call"] == "closest":
        return sc.cast_rays(st["org"], st["dir"], st["tnear"], st["tfar"], normals=True)
    if case["call"] == "records":
        return sc.cast_ray_records(st["org"], st["dir"], st["tnear"], st["tfar"])
    return sc.occluded(st["org"], st["dir"], st["tnear"], st["tfar"])


def _run_render(case, st):
    r = st["renderer"]
    r.reset()
    r.render(case["spp"])
    w, h = case["width"], case["height"]
    if w * h <= 1 << 16:   # a small preview is shown from host memory
        return {"raw": r.raw(), "progress": r.current_progress(), "normals": r.current_normals()}
    return {"raw": _device_buffer(r, "raw", (h, w, 3)), "progress": _device_buffer(r, "progress", (h, w, 4)),
            "albedos": _device_buffer(r, "albedos", (h, w, 4)), "normals": _device_buffer(r, "normals", (h, w, 4)),
            "depths": _device_buffer(r, "depths", (h, w, 4))}


def _run_batch(case, st):
    return render_batch(st["ctx"], st["jobs"])[0]


def _run_infer(case, st):
    A.check(A.lib().crt_nrc_infer(st["nrc"].handle, C.c_void_p(st["queries"].data_ptr()), case["n"],
                                  C.c_void_p(st["out"].data_ptr()), A.CRT_MEM_DEVICE))
    return st["out"]


def _run_gradient(case, st):
    loss = C.c_float()
    A.check(A.lib().crt_nrc_gradient(st["nrc"].handle, C.c_void_p(st["queries"].data_ptr()),
                                     C.c_void_p(st["targets"].data_ptr()), case["n"], A.vptr(st["grad"]),
                                     C.byref(loss), A.CRT_MEM_DEVICE))
    return {"grad": st["grad"], "loss": loss.value}


def _run_finish(case, st):
    col, nrm, alb, shown = st["images"]
    post = dict(bloom=True, gray=bool(case["gray"]), tonemap=True, tonemap_type=case["tonemap"], exposure=1.2,
                full_coverage=bool(case["full"]))
    if case["memory"] == "host":
        return {"denoised": denoise(st["ctx"], col, nrm, alb, levels=case["levels"]),
                "shown": post_process(st["ctx"], shown, **post)}
    L, h, w = A.lib(), case["height"], case["width"]

    def ptr(t):
        return C.c_void_p(t.data_ptr())

    o = A.DenoiseOptions(case["levels"], 2.0, 0.2, 0.2)
    A.check(L.crt_denoise(st["ctx"].handle, C.byref(o), ptr(col), ptr(nrm), ptr(alb), ptr(st["denoised"]), w, h,
                          A.CRT_MEM_DEVICE))
    p = A.PostOptions()
    L.crt_post_options_default(C.byref(p))
    p.bloom, p.gray_scale, p.tonemapping, p.tonemapping_type = 1, case["gray"], 1, case["tonemap"]
    p.exposure, p.full_coverage = 1.2, case["full"]
    A.check(L.crt_post_process(st["ctx"].handle, C.byref(p), ptr(shown), ptr(st["shown"]), w, h, A.CRT_MEM_DEVICE))
    return {"denoised": st["denoised"], "shown": st["shown"]}


def _run_load(case, st):
    sc = Scene(st["ctx"])
    sc.add_model(st["spec"])
    sc.set_camera(st["spec"].camera)
    sc.commit()
    hits = sc.cast_rays(st["org"], st["dir"], normals=True)
    sc.close()
    return hits


# ---- work ---------------------------------------------------------------------------------

def work(case):
    """Bytes: every input read once and every output written once (a ray 32 B, a hit field
    4 B, a triangle 36 B, a pixel-sample's running sum 24 B).  Operations: per ray a descent
    of about log2(triangles) box tests of 20 flops and two triangle tests of 50."""
    kind = case["kind"]
    if kind == "query":
        n, tris = case["n"], case["tris"]
        out = {"closest": 36, "records": 48, "occluded": 1}[case["call"]]
        return {"bytes": n * (32 + out) + min(36 * tris, 36 * n), "flops": _ray_flops(tris) * n}
    if kind == "render":
        px = case["width"] * case["height"] * case["spp"]
        tris = {"cornell": 36, "cutout": 44}.get(case["scene"], case["tris"])
        rays = 2 * px
        return {"bytes": 24 * px + 48 * rays + 36 * tris + 64 * case["width"] * case["height"],
                "flops": _ray_flops(tris) * rays}
    if kind == "batch":
        px = case["jobs"] * case["edge"] ** 2 * case["spp"] // 3
        return {"bytes": (24 + 96) * px + 36 * case["jobs"] * case["tris"], "flops": 2 * px * _ray_flops(case["tris"])}
    params = sum(k * n for k, n in LAYERS)
    if kind == "infer":
        return {"bytes": 64 * case["n"] + 2 * params, "flops": 2 * params * case["n"]}
    if kind == "gradient":
        return {"bytes": 64 * case["n"] + 6 * params, "flops": 6 * params * case["n"]}
    if kind == "finish":
        px = case["width"] * case["height"]
        return {"bytes": (64 + 32) * px, "flops": (case["levels"] * 25 * 30 + 10 * 15 * 6) * px}
    return {"bytes": 36 * case["tris"] * 2 + 68 * case["n"], "flops": 200 * case["tris"] + _ray_flops(case["tris"]) * case["n"]}


def _ray_flops(tris):
    return int(20 * 2 * math.log2(max(tris, 2)) + 100)


# ---- exact --------------------------------------------------------------------------------

def exact(case, seed):
    kind = case["kind"]
    if kind == "query":
        if case["call"] == "occluded" or case["n"] * case["tris"] * case["instances"] > 10_000_000_000:
            return None
        return _exact_query(case, *_query_inputs(case, seed))
    if kind == "load":
        verts, rays = _load_inputs(case, seed)
        full = _exact_query({"call": "closest", "memory": "host", "instances": 1}, verts, None, rays)
        return full
    if kind == "infer":
        ws, g = _net(seed)
        q = _cache_queries(g, case["n"])
        ws = [w.to(F64) for w in ws]
        return torch.cat([_mlp(q[i:i + 262_144], ws)[:, :3] for i in range(0, case["n"], 262_144)])
    if kind == "gradient":
        return _exact_gradient(case, seed)
    if kind == "finish":
        return _exact_finish(case, seed)
    return None   # whole renders: a path tracer's decisions do not carry over to FP64


def _exact_query(case, verts, inst, rays):
    """Closest hits by brute force over all (placed) triangles."""
    tri = verts.to(F64).reshape(-1, 3, 3)
    ntri = tri.shape[0]
    world = tri
    if inst is not None:
        m = torch.as_tensor(inst, device=DEV).to(F64).reshape(-1, 4, 4)   # m[i] is the transposed matrix
        world = torch.einsum("tcx,ixy->itcy", tri, m[:, :3, :3]) + m[:, None, None, 3, :3]
        world = world.reshape(-1, 3, 3)
    r = rays.to(F64)
    o, d, tn, tf = r[0:3].T, r[3:6].T, r[6], r[7]
    records = case["call"] == "records"
    if records:
        d = d / d.norm(dim=1, keepdim=True)
    v0, e1, e2 = world[:, 0], world[:, 1] - world[:, 0], world[:, 2] - world[:, 0]
    n, total = o.shape[0], world.shape[0]
    best_t = torch.empty(n, device=DEV, dtype=F64)
    best_k = torch.empty(n, device=DEV, dtype=torch.int64)
    nrm = torch.linalg.cross(e1, e2)
    step = max(1, (1 << 24) // total)
    for b in range(0, n, step):
        oo, dd = o[b:b + step], d[b:b + step]
        # Moeller-Trumbore with the products split into per-triangle and per-ray parts
        det = -(dd @ nrm.T)
        s = [oo[:, None, k] - v0[None, :, k] for k in range(3)]
        q = [s[(k + 1) % 3] * dd[:, None, (k + 2) % 3] - s[(k + 2) % 3] * dd[:, None, (k + 1) % 3] for k in range(3)]
        u = (q[0] * e2[None, :, 0] + q[1] * e2[None, :, 1] + q[2] * e2[None, :, 2]) / det
        v = -(q[0] * e1[None, :, 0] + q[1] * e1[None, :, 1] + q[2] * e1[None, :, 2]) / det
        t = (s[0] * nrm[None, :, 0] + s[1] * nrm[None, :, 1] + s[2] * nrm[None, :, 2]) / det
        ok = (det != 0) & (u >= 0) & (v >= 0) & (u + v <= 1) & (t > tn[b:b + step, None]) & (t <= tf[b:b + step, None])
        t = torch.where(ok, t, torch.full_like(t, math.inf))
        best_t[b:b + step], best_k[b:b + step] = t.min(dim=1)
    hit = torch.isfinite(best_t)
    k = best_k
    det = -(d * nrm[k]).sum(1)
    s = o - v0[k]
    q = torch.linalg.cross(s, d)
    zero = torch.zeros_like(best_t)
    u = torch.where(hit, (q * e2[k]).sum(1) / det, zero)
    v = torch.where(hit, -(q * e1[k]).sum(1) / det, zero)
    prim = k % ntri
    ob = tri[prim]
    ng = torch.linalg.cross(ob[:, 1] - ob[:, 0], ob[:, 2] - ob[:, 0])
    if records:
        ng = ng / ng.norm(dim=1, keepdim=True)
        p = torch.where(hit[:, None], o + d * torch.where(hit, best_t, zero)[:, None], zero[:, None].expand(-1, 3))
    ng = torch.where(hit[:, None], ng, torch.zeros_like(ng))
    if records:
        out = {"distance": best_t, "u": zero, "v": zero, "n_x": ng[:, 0], "n_y": ng[:, 1], "n_z": ng[:, 2],
               "p_x": p[:, 0], "p_y": p[:, 1], "p_z": p[:, 2]}
        keys = A.RECORD_FIELDS
    else:
        out = {"t": best_t, "u": u, "v": v, "ng_x": ng[:, 0], "ng_y": ng[:, 1], "ng_z": ng[:, 2]}
        keys = HIT_KEYS if case["memory"] == "device" else ("t", "u", "v", "prim_id", "geom_id", "inst_id", "ng_x",
                                                            "ng_y", "ng_z")
    return {key: out.get(key) for key in keys}


def _mlp(q, ws):
    """The cache's network in FP64: 12-frequency sin / cos of the position, the other ten
    inputs, a constant 1, zero padding; five ReLU layers and a linear one."""
    q = q.to(F64)
    arg = q[:, :3, None] * (math.pi * 2.0 ** torch.arange(12, device=DEV, dtype=F64))
    enc = torch.stack([torch.sin(arg), torch.cos(arg)], 3).reshape(q.shape[0], 72)
    x = torch.cat([enc, q[:, 3:], torch.ones((q.shape[0], 1), device=DEV, dtype=F64),
                   torch.zeros((q.shape[0], 13), device=DEV, dtype=F64)], 1)
    for w in ws[:-1]:
        x = torch.relu(x @ w)
    return x @ ws[-1]


def _exact_gradient(case, seed):
    ws, g = _net(seed)
    q = _cache_queries(g, case["n"])
    t = _cache_targets(g, case["n"]).to(F64)
    ws = [w.to(F64).requires_grad_(True) for w in ws]
    with torch.enable_grad():
        y = _mlp(q, ws)[:, :3]
        loss = ((y - t) ** 2 / (y.detach() ** 2 + 0.01)).sum() / (3.0 * case["n"])
        grads = torch.autograd.grad(loss, ws)
    return {"grad": torch.cat([x.reshape(-1) for x in grads]), "loss": float(loss.detach())}


def _exact_finish(case, seed):
    col, nrm, alb, shown = (x.to(F64) for x in _finish_inputs(case, seed))
    h, w = case["height"], case["width"]
    kern = (3.0 / 8.0, 1.0 / 4.0, 1.0 / 16.0)
    src = col[..., :3]
    n3, a3 = nrm[..., :3], alb[..., :3]
    for level in range(case["levels"]):
        step, sc = 1 << level, 2.0 * 2.0 ** -level
        acc, wsum = torch.zeros_like(src), torch.zeros((h, w, 1), device=DEV, dtype=F64)
        for dy in range(-2, 3):
            for dx in range(-2, 3):
                oy, ox = dy * step, dx * step
                if abs(oy) >= h or abs(ox) >= w:
                    continue
                ya, yb, xa, xb = max(0, -oy), h - max(0, oy), max(0, -ox), w - max(0, ox)
                here = (slice(ya, yb), slice(xa, xb))
                there = (slice(ya + oy, yb + oy), slice(xa + ox, xb + ox))
                dc = ((src[there] - src[here]) ** 2).sum(2, keepdim=True)
                dn = ((n3[there] - n3[here]) ** 2).sum(2, keepdim=True)
                da = ((a3[there] - a3[here]) ** 2).sum(2, keepdim=True)
                wt = kern[abs(dx)] * kern[abs(dy)] * torch.exp(-(dc / sc ** 2 + dn / 0.04 + da / 0.04))
                acc[here] += wt * src[there]
                wsum[here] += wt
        src = acc / wsum
    one = torch.ones((h, w, 1), device=DEV, dtype=F64)
    return {"denoised": torch.cat([src, one], 2), "shown": _exact_post(case, shown, h, w)}


def _exact_post(case, img, h, w):
    blur = (0.19744746769063704, 0.1746973469158936, 0.12099884565428047, 0.06560233156931679, 0.027839605612666265,
            0.009246250740395456, 0.002403157286908872, 0.00048872837522002)
    cw, ch = (w, h) if case["full"] else (w // 8 * 8, h // 8 * 8)
    rgb = img[..., :3]
    luma = rgb @ torch.tensor([0.2126, 0.7152, 0.0722], device=DEV, dtype=F64)
    b = torch.where((luma < 0.7)[..., None], torch.zeros_like(rgb), rgb)
    for i in range(10):
        axis = 1 if i % 2 == 0 else 0
        size = w if axis == 1 else h
        out = b * blur[0]
        for k in range(1, min(8, size)):
            head, tail = b.narrow(axis, 0, size - k), b.narrow(axis, k, size - k)
            out.narrow(axis, 0, size - k).add_(tail * blur[k])
            out.narrow(axis, k, size - k).add_(head * blur[k])
        out[ch:] = 0.0
        out[:, cw:] = 0.0
        b = out
    c = rgb + b
    if case["gray"]:
        c = (c @ torch.tensor([0.2126, 0.7162, 0.0722], device=DEV, dtype=F64))[..., None].expand(-1, -1, 3)
    c = c * float(np.float32(1.2))
    ig = 1.0 / float(np.float32(2.2))
    kind = case["tonemap"]
    if kind == 0:
        c = c ** ig
    elif kind == 1:
        c = (c / (c + 1.0)) ** ig
    elif kind == 2:
        x = torch.clamp(c - 0.004, min=0.0)
        c = (x * (6.2 * x + 0.5)) / (x * (6.2 * x + 1.7) + 0.06)
    else:
        def curve(x):
            return (x * (0.15 * x + 0.05) + 0.004) / (x * (0.15 * x + 0.5) + 0.06) - 0.02 / 0.30

        c = (curve(2.0 * c) / curve(torch.tensor(11.2, device=DEV, dtype=F64))) ** ig
    out = torch.cat([c, torch.ones((h, w, 1), device=DEV, dtype=F64)], 2)
    out[ch:] = 0.0
    out[:, cw:] = 0.0
    return out
