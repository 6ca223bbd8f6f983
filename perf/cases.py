"""Workloads of the triangle ray-query library, as programs that use it run them.

A case is a dict of plain values; its "op" says which calls a pass makes:

  query    rtcgIntersect1MAsync / rtcgOccluded1MAsync over records in GPU memory
  host     rtcIntersect1M over records in host memory
  single   rtcIntersect1 on one record in host memory
  frame    new vertices in host memory, rtcCommitScene, then a closest-hit query
  inst     a two-level scene: closest hits, then one shadow ray per record
  batch    many scenes committed together, all their streams in one graph launch

Every pass starts from fresh records (a copy of the caller's generated rays),
because a query updates the records in place.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "embree-aarch64_amd"))

import rtcore as R  # noqa: E402

QUALITY = {"low": R.RTC_BUILD_QUALITY_LOW, "medium": R.RTC_BUILD_QUALITY_MEDIUM, "high": R.RTC_BUILD_QUALITY_HIGH}
PAIRS_EXACT = 1 << 33  # ray-triangle pairs that exact() tests one by one in double precision

_kept = {}


def device():
    """The one RTCDevice of the process, with the default settings."""
    if "device" not in _kept:
        _kept["device"] = R.Device("")
    return _kept["device"]


def stream():
    """The stream the program's rays are made and traced on."""
    if "stream" not in _kept:
        _kept["stream"] = torch.cuda.Stream()
    return _kept["stream"]


# ------------------------------------------------------------------ cases --

def listed():
    return [
        # a picking ray: the smallest call of a program written for the CPU library
        {"name": "single_sphere", "op": "single", "mesh": "sphere", "size": 64, "quality": "medium", "robust": False},
        # a probe update or a small wavefront queue: latency, a launch that cannot fill the GPU
        {"name": "probes_terrain", "op": "query", "mesh": "terrain", "size": 257, "rays": "camera", "width": 37,
         "height": 29, "kind": "closest", "quality": "medium", "robust": False},
        # the primary rays of a full-HD frame over a 2.1 M triangle terrain
        {"name": "camera_terrain", "op": "query", "mesh": "terrain", "size": 1025, "rays": "camera", "width": 1920,
         "height": 1080, "kind": "closest", "quality": "medium", "robust": False},
        # its cosine-distributed bounces
        {"name": "bounce_terrain", "op": "query", "mesh": "terrain", "size": 1025, "rays": "bounce", "width": 1531,
         "height": 977, "kind": "closest", "quality": "medium", "robust": False},
        # incoherent closest hits, the workload of the benchmark
        {"name": "random_soup", "op": "query", "mesh": "soup", "size": 1 << 20, "rays": "random", "width": 4096,
         "height": 4096, "kind": "closest", "quality": "medium", "robust": False},
        # short occlusion rays in the same scene (ambient occlusion)
        {"name": "occluded_soup", "op": "query", "mesh": "soup", "size": 1 << 20, "rays": "random", "width": 4096,
         "height": 2048, "kind": "occluded", "quality": "medium", "robust": False},
        # a scene with the robust flag, ragged sizes
        {"name": "robust_soup", "op": "query", "mesh": "soup", "size": 250007, "rays": "random", "width": 1999,
         "height": 1051, "kind": "closest", "quality": "medium", "robust": True},
        # a program that keeps its records in host memory
        {"name": "host_sphere", "op": "host", "mesh": "sphere", "size": 251, "width": 2048, "height": 1024,
         "quality": "medium", "robust": False},
        # a deforming mesh of an interactive program: commit and trace every frame
        {"name": "frame_small", "op": "frame", "mesh": "sphere", "size": 71, "width": 256, "height": 256,
         "quality": "low", "robust": False},
        # a large scene committed at the default quality, then one frame
        {"name": "frame_soup", "op": "frame", "mesh": "soup", "size": 1 << 20, "width": 1024, "height": 1024,
         "quality": "medium", "robust": False},
        # 10,000 instances of five meshes, camera and shadow rays
        {"name": "instances", "op": "inst", "size": 10000, "scale": 0.2, "width": 2048, "height": 1024},
        # many small scenes served together
        {"name": "batch_spheres", "op": "batch", "size": 64, "tris": 200000, "width": 131072},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mesh(rng, most):
    """A mesh kind and its size parameter, up to about `most` triangles."""
    kind = rng.choice(["sphere", "terrain", "soup"])
    tris = _log_int(rng, 1000, most)
    if kind == "sphere":
        return kind, max(4, int(0.5 + math.sqrt(tris / 4.0)))
    if kind == "terrain":
        return kind, max(3, int(math.sqrt(tris / 2.0)) + 1)
    return kind, tris


def draw(rng):
    op = rng.choice(["query", "query", "query", "query", "host", "single", "frame", "frame", "inst", "batch"])
    if op == "inst":
        w, h = _image(rng, 1 << 10, 1 << 21)
        return {"op": op, "size": _log_int(rng, 10, 10000), "scale": round(rng.uniform(0.05, 0.2), 3), "width": w,
                "height": h}
    if op == "batch":
        return {"op": op, "size": _log_int(rng, 2, 64), "tris": _log_int(rng, 2000, 200000),
                "width": _log_int(rng, 500, 131072)}
    kind, size = _mesh(rng, 1 << 20)
    case = {"op": op, "mesh": kind, "size": size}
    if op == "query":
        case["rays"] = rng.choice(["camera", "bounce", "random"])
        case["width"], case["height"] = _image(rng, 1, 1 << 23)
        case["kind"] = rng.choice(["closest", "closest", "occluded"])
        case["quality"] = rng.choice(["low", "medium", "medium", "high"])
        case["robust"] = rng.random() < 0.25
    elif op == "host":
        case["width"], case["height"] = _image(rng, 1, 1 << 21)
        case["quality"], case["robust"] = "medium", rng.random() < 0.25
    elif op == "single":
        case["quality"], case["robust"] = "medium", rng.random() < 0.25
    else:
        case["width"], case["height"] = _image(rng, 64, 1 << 20)
        case["quality"] = rng.choice(["low", "medium", "medium", "high"])
        case["robust"] = rng.random() < 0.25
    return case


def _image(rng, lo, hi):
    n = _log_int(rng, lo, hi)
    w = max(1, int(math.sqrt(n * rng.uniform(0.8, 2.0))))
    return w, max(1, n // w)


# ----------------------------------------------------------------- inputs --

def mesh(case, seed):
    """Vertices and indices of a case's mesh."""
    kind, size = case["mesh"], case["size"]
    if kind == "sphere":
        return R.gen_displaced_sphere(size, seed=seed + 1, amplitude=0.1)
    if kind == "terrain":
        return R.gen_heightfield(size, seed=seed + 1, amplitude=0.2, octaves=6)
    # triangles of half extent 0.005 at 2^20 of them, larger where there are fewer (the same share of the volume)
    rng = np.random.default_rng(seed + 1)
    h = np.float32(0.005 * (float(1 << 20) / size) ** (1.0 / 3.0))
    v = (rng.random((size, 3, 3), dtype=np.float32) * 2 - 1) * h
    v += rng.random((size, 1, 3), dtype=np.float32)
    return v.reshape(-1, 3), np.arange(3 * size, dtype=np.uint32).reshape(-1, 3)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + 13)
    return g


def records(org, dirs, tfar, hit):
    """RTCRayHit (hit) or RTCRay records as a float32 tensor [n, 20 or 12]."""
    n = org.shape[0]
    r = torch.zeros(n, 20 if hit else 12, device="cuda")
    r[:, 0:3], r[:, 4:7], r[:, 8] = org, dirs, tfar
    words = r.view(torch.int32)
    words[:, 9] = -1
    words[:, 10] = torch.arange(n, device="cuda", dtype=torch.int32)
    if hit:
        words[:, 17:20] = -1
    return r


def _unit(v):
    return v / v.norm(dim=-1, keepdim=True)


def camera_rays(w, h, org, target, up, fov, g):
    """A pinhole camera's rays, one jittered sample in each pixel."""
    o, t, u = (torch.tensor(x, device="cuda") for x in (org, target, up))
    z = _unit(t - o)
    x = _unit(torch.linalg.cross(z, u))
    y = torch.linalg.cross(x, z)
    s = math.tan(math.radians(fov) / 2)
    j = torch.rand(h, w, 2, device="cuda", generator=g)
    px = ((torch.arange(w, device="cuda") + j[..., 0]) / w * 2 - 1) * s * (w / h)
    py = (1 - (torch.arange(h, device="cuda")[:, None] + j[..., 1]) / h * 2) * s
    d = _unit(z + px[..., None] * x + py[..., None] * y).reshape(-1, 3)
    return o.expand_as(d), d


def _sphere_dirs(n, g):
    z = torch.rand(n, device="cuda", generator=g) * 2 - 1
    a = torch.rand(n, device="cuda", generator=g) * (2 * math.pi)
    s = (1 - z * z).clamp_min(0).sqrt()
    return torch.stack([s * a.cos(), s * a.sin(), z], 1)


VIEWS = {  # camera position, target, up and field of view for each mesh
    "terrain": ((0.5, -0.35, 0.5), (0.5, 0.55, 0.0), (0.0, 0.0, 1.0), 50.0),
    "sphere": ((0.0, 0.0, 3.0), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 45.0),
    "soup": ((0.5, 0.5, -1.2), (0.5, 0.5, 0.5), (0.0, 1.0, 0.0), 50.0),
}


def _view(kind, seed):
    org, target, up, fov = VIEWS[kind]
    rng = np.random.default_rng(seed + 5)
    return tuple(float(a + b) for a, b in zip(org, rng.uniform(-0.05, 0.05, 3))), target, up, fov


def host_rays(case, seed):
    """A camera's records, or the one through a point near an image's middle."""
    org, target, up, fov = _view(case["mesh"], seed)
    if case["op"] == "single":
        return records(*camera_rays(1, 1, org, target, up, fov / 3, _gen(seed)), math.inf, True)
    return records(*camera_rays(case["width"], case["height"], org, target, up, fov, _gen(seed)), math.inf, True)


def rays_of(case, scene, seed):
    """The records that a query case traces."""
    g, w, h = _gen(seed), case["width"], case["height"]
    n, closest = w * h, case["kind"] == "closest"
    if case["rays"] == "random":  # origins in the mesh's volume, directions over the sphere
        lo, hi = (-1.0, 1.0) if case["mesh"] == "sphere" else (0.0, 1.0)
        org = torch.rand(n, 3, device="cuda", generator=g) * (hi - lo) + lo
        return records(org, _sphere_dirs(n, g), math.inf if closest else 0.1, closest)
    org, dirs = camera_rays(w, h, *_view(case["mesh"], seed), g)
    if case["rays"] == "bounce":
        first = records(org, dirs, math.inf, True)
        trace(scene, first, True)
        stream().synchronize()
        first = first[first.view(torch.int32)[:, 18] != -1]
        if len(first) == 0:
            return records(org, dirs, math.inf if closest else 10.0, closest)
        first = first[torch.arange(n, device="cuda") % len(first)]
        normal = _unit(first[:, 12:15])
        normal = torch.where((normal * first[:, 4:7]).sum(1, keepdim=True) > 0, -normal, normal)
        org = first[:, 0:3] + first[:, 8:9] * first[:, 4:7] + 1e-4 * normal
        dirs = _unit(normal + 0.999 * _sphere_dirs(n, g))
    return records(org, dirs, math.inf if closest else 10.0, closest)


def trace(scene, recs, closest):
    """Queues a query over device records on the program's stream."""
    s = stream()
    s.wait_stream(torch.cuda.current_stream())
    call = R.lib().rtcgIntersect1MAsync if closest else R.lib().rtcgOccluded1MAsync
    call(scene.h, ctypes.byref(R.init_context()), recs.data_ptr(), len(recs), recs.shape[1] * 4, s.cuda_stream)


def fields(recs):
    """The output fields of closest-hit records (or the one of occlusion records), as views."""
    if recs.shape[1] == 12:
        return {"tfar": recs[:, 8]}
    words = recs.view(torch.int32) if isinstance(recs, torch.Tensor) else recs.view(np.int32)
    return {"tfar": recs[:, 8], "Ng": recs[:, 12:15], "uv": recs[:, 15:17], "ids": words[:, 17:20]}


class State:
    """What a program holds: scenes and records. Gives the scenes back when dropped."""

    def __init__(self):
        self.scenes, self.graph, self.ctx = [], None, R.init_context()

    def __del__(self):
        torch.cuda.synchronize()
        if self.graph:
            R.lib().rtcgReleaseBatchGraph(self.graph)
        for s in self.scenes:
            s.release()


def _scene(case, v, ix, shared=False):
    flags = R.RTC_SCENE_FLAG_ROBUST if case["robust"] else 0
    return R.Scene(device(), [(v, ix)], quality=QUALITY[case["quality"]], flags=flags, shared=shared)


def prepare(case, seed):
    st = State()
    st.op = op = case["op"]
    if op == "inst":
        _prepare_instances(st, case, seed)
    elif op == "batch":
        _prepare_batch(st, case, seed)
    elif op == "frame":
        _prepare_frame(st, case, seed)
    else:
        v, ix = mesh(case, seed)
        st.scenes = [_scene(case, v, ix).commit()]
        if op == "query":
            st.closest = case["kind"] == "closest"
            st.src = rays_of(case, st.scenes[0], seed)
            st.recs = st.src.clone()
            st.out = fields(st.recs)
        else:
            st.src = host_rays(case, seed).cpu()
            st.recs = st.src.clone()
            st.out = fields(st.recs.numpy())
    torch.cuda.synchronize()
    return st


def _prepare_frame(st, case, seed):
    """Geometry in the caller's own buffers (padded to 16 readable bytes past
    the last vertex), which the program rewrites between the commits."""
    v, ix = mesh(case, seed)
    st.verts = np.zeros((len(v) + 1, 3), np.float32)
    st.verts[:-1], st.index = v, np.ascontiguousarray(ix)
    L, d = R.lib(), device()
    sc = R.Scene(d, quality=QUALITY[case["quality"]], flags=R.RTC_SCENE_FLAG_ROBUST if case["robust"] else 0)
    g = L.rtcNewGeometry(d.h, R.RTC_GEOMETRY_TYPE_TRIANGLE)
    L.rtcSetSharedGeometryBuffer(g, R.RTC_BUFFER_TYPE_VERTEX, 0, R.RTC_FORMAT_FLOAT3, st.verts.ctypes.data, 0, 12,
                                 len(v))
    L.rtcSetSharedGeometryBuffer(g, R.RTC_BUFFER_TYPE_INDEX, 0, R.RTC_FORMAT_UINT3, st.index.ctypes.data, 0, 12,
                                 len(ix))
    L.rtcCommitGeometry(g)
    L.rtcAttachGeometry(sc.h, g)
    L.rtcReleaseGeometry(g)  # the scene keeps it
    st.geom, st.scenes, st.closest = g, [sc], True
    st.src = host_rays(case, seed)
    st.recs = st.src.clone()
    st.out = fields(st.recs)


def _prepare_instances(st, case, seed):
    d, scale = device(), case["scale"]
    a = max(4, int(500 * math.sqrt(scale)))
    b = max(5, int(708 * math.sqrt(scale)))
    meshes = R.instance_workload(seed=seed + 11, sizes=(a, max(4, a // 2), b, max(5, b // 2), max(5, b // 3)))
    bases = [R.Scene(d, [m]).commit() for m in meshes]
    # the instances keep their density: 10,000 of them fill [-50, 50]^3
    extent = 50.0 * (case["size"] / 10000.0) ** (1.0 / 3.0)
    top = R.Scene(d)
    for k, m in enumerate(R.random_transforms(case["size"], seed=seed + 5, extent=extent)):
        top.add_instance(bases[k % len(bases)], m)
    top.commit()
    st.scenes = [top] + bases
    g = _gen(seed)
    org, dirs = camera_rays(case["width"], case["height"], (0.0, 0.0, 2.6 * extent), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0),
                            45.0, g)
    st.src = records(org, dirs, math.inf, True)
    st.recs = st.src.clone()
    trace(top, st.recs, True)
    stream().synchronize()
    # shadow rays from the hit points (where a ray missed: from beside the
    # centre) to a light above; the light sits at t = 1
    t = torch.where(torch.isinf(st.recs[:, 8]), torch.full_like(st.recs[:, 8], 2.6 * extent), st.recs[:, 8])
    p = org + t[:, None] * dirs
    light = torch.tensor([0.0, 2.0 * extent, 0.0], device="cuda")
    st.shadow_src = records(p, light - p, 1.0, False)
    st.shadow_src[:, 3] = 1e-4
    st.shadow = st.shadow_src.clone()
    st.out = {"closest": fields(st.recs), "shadow": fields(st.shadow)}


def _streams(case):
    """(ring count, rays) of each scene of a batch, log-uniform up to the case's sizes."""
    return [(p, r) for p, _, r in R.batch_workload(case["size"], tri_range=(1e3, case["tris"]),
                                                   ray_range=(min(500, case["width"]), case["width"]))]


def _prepare_batch(st, case, seed):
    d, streams, g = device(), _streams(case), _gen(seed)
    st.scenes = [R.Scene(d, [R.gen_displaced_sphere(p, seed=seed + i)]) for i, (p, _) in enumerate(streams)]
    R.commit_scenes(st.scenes)
    n = sum(r for _, r in streams)
    org = 2.0 * _sphere_dirs(n, g)
    inside = _sphere_dirs(n, g) * torch.rand(n, 1, device="cuda", generator=g) ** (1.0 / 3.0)
    st.src = records(org, _unit(inside - org), math.inf, True)
    st.recs = st.src.clone()
    items, at = [], 0
    for sc, (_, r) in zip(st.scenes, streams):
        items.append((sc, st.recs.data_ptr() + 80 * at, r, 80))
        at += r
    st.items = R.batch_items(items)
    st.graph = R.lib().rtcgNewBatchGraph(st.items.ctypes.data, len(st.items), 0)
    d.check("rtcgNewBatchGraph")
    st.out = fields(st.recs)


# ------------------------------------------------------------------- pass --

def run(st):
    L = R.lib()
    if st.op in ("single", "host"):
        st.recs.copy_(st.src)
        if st.op == "single":
            L.rtcIntersect1(st.scenes[0].h, ctypes.byref(st.ctx), st.recs.data_ptr())
        else:
            L.rtcIntersect1M(st.scenes[0].h, ctypes.byref(st.ctx), st.recs.data_ptr(), len(st.recs), 80)
        return st.out
    s = stream()
    with torch.cuda.stream(s):
        if st.op == "frame":
            L.rtcUpdateGeometryBuffer(st.geom, R.RTC_BUFFER_TYPE_VERTEX, 0)
            L.rtcCommitGeometry(st.geom)
            L.rtcCommitScene(st.scenes[0].h)
        st.recs.copy_(st.src)
        if st.op == "batch":
            L.rtcgLaunchBatchGraph(st.graph, s.cuda_stream)
            return st.out
        call = L.rtcgOccluded1MAsync if st.recs.shape[1] == 12 else L.rtcgIntersect1MAsync
        call(st.scenes[0].h, ctypes.byref(st.ctx), st.recs.data_ptr(), len(st.recs), st.recs.shape[1] * 4,
             s.cuda_stream)
        if st.op == "inst":
            st.shadow.copy_(st.shadow_src)
            L.rtcgOccluded1MAsync(st.scenes[0].h, ctypes.byref(st.ctx), st.shadow.data_ptr(), len(st.shadow), 48,
                                  s.cuda_stream)
    return st.out


# ------------------------------------------------------------------- work --

def _tris(case):
    n = case["size"]
    return {"sphere": 4 * n * (n - 1), "terrain": 2 * (n - 1) ** 2, "soup": n}[case["mesh"]]


def work(case):
    """Rays read (36 B) and results written (36 B closest hit, 4 B occlusion)
    once, geometry read once where a ray can reach it (48 B a triangle), and,
    for a commit, the triangles read and their records written. Operations: a
    ray tests one triangle (about 50) and the 8 boxes (about 12 each) of each
    node on one path from the root."""
    def path(tris):
        return 50 + 96 * max(1.0, math.log(max(tris, 8), 8))

    if case["op"] == "inst":
        n, s = case["width"] * case["height"], case["scale"]
        return {"bytes": n * (72 + 40) + case["size"] * 64 + 2.5e6 * s * 48, "flops": 2.0 * n * path(5e5 * s)}
    if case["op"] == "batch":
        lo, hi = min(500, case["width"]), case["width"]
        rays = case["size"] * ((hi - lo) / math.log(hi / lo) if hi > lo else hi)
        tris = case["size"] * (case["tris"] - 1e3) / math.log(case["tris"] / 1e3)
        return {"bytes": rays * 72 + tris * 48, "flops": rays * path(case["tris"])}
    tris = _tris(case)
    n = 1 if case["op"] == "single" else case["width"] * case["height"]
    ray = 40 if case.get("kind") == "occluded" else 72
    data = n * ray + min(tris, 8 * n) * 48
    if case["op"] == "frame":
        data += tris * (48 + 48 + 32)
    return {"bytes": data, "flops": n * path(tris) + (tris * 40.0 if case["op"] == "frame" else 0.0)}


# ------------------------------------------------------------------ exact --

def exact(case, seed):
    """The nearest hits of a closest-hit case in double precision, by testing
    every triangle; None where that is too much."""
    if case["op"] in ("inst", "batch") or case.get("kind") == "occluded":
        return None
    n = 1 if case["op"] == "single" else case["width"] * case["height"]
    if n * _tris(case) > PAIRS_EXACT or case.get("rays") == "bounce":
        return None
    v, ix = mesh(case, seed)
    rec = rays_of(case, None, seed) if case["op"] == "query" else host_rays(case, seed)
    p = torch.from_numpy(v).double().cuda()[torch.from_numpy(ix.astype(np.int64)).cuda()]
    v0, e1, e2 = p[:, 0], p[:, 0] - p[:, 1], p[:, 2] - p[:, 0]
    normal = torch.linalg.cross(e2, e1)
    out = {"tfar": rec[:, 8].double(), "Ng": torch.zeros(n, 3, dtype=torch.float64, device="cuda"),
           "uv": torch.zeros(n, 2, dtype=torch.float64, device="cuda"), "ids": None}
    step = max(1, (1 << 25) // len(v0))
    for a in range(0, n, step):
        o, d = rec[a:a + step, None, 0:3].double(), rec[a:a + step, None, 4:7].double()
        c = v0[None] - o
        r = torch.linalg.cross(c, d.expand_as(c))
        den = (normal[None] * d).sum(-1)
        u, w = (r * e2[None]).sum(-1) / den, (r * e1[None]).sum(-1) / den
        t = (normal[None] * c).sum(-1) / den
        t = torch.where((den != 0) & (u >= 0) & (w >= 0) & (u + w <= 1) & (t > 0), t, math.inf)
        best, k = t.min(1)
        hit = torch.isfinite(best)
        rows, k = torch.arange(len(k), device="cuda")[hit], k[hit]
        out["tfar"][a:a + step] = best
        out["Ng"][a + rows] = normal[k]
        out["uv"][a + rows] = torch.stack([u[rows, k], w[rows, k]], 1)
    return out
