"""The work this framework is used for, as measurable cases through its public entry points.

A case names a `kind` (which entry points one pass goes through) and its sizes:

  closest    Accel.trace_closest over a resident scene: camera and bounce rays of a renderer,
             visibility and distance queries of a simulation
  any        Accel.trace_any over segments between scene points (shadow and line-of-sight rays)
  frame      the geometry is new in every pass: Mesh.build + Accel.build + Accel.trace_closest, with
             either AccelOption hint (the default FAST_TRACE, or FAST_BUILD)
  animate    deforming geometry: new vertices into the mesh's buffer, Mesh.build as an update
             (allow_update), Accel.build, Accel.trace_closest
  instances  a scene of instanced meshes of which some move: set_transform_on_update, Accel.build,
             one Accel.trace_batched over ray batches of different sizes
  query      Accel.query (traverse with surface and procedural callbacks) over triangles with a
             cutout and AABBs with spheres
  render     Accel.pathtrace of the closed room, as wavefront or megakernel
  shader     the path tracer written in the Python DSL, compiled at run time, one dispatch
  serve      requests of different sizes submitted to a render server and drained

Sizes are those of the repository's benchmark workloads, tests and golden fixtures or lie between
them. Scenes live in [0, 100]^3: triangle soups whose triangles shrink as their number grows (the
benchmark's soup at 16,777,216 triangles), and closed wavy spheres; the renders use the
benchmark's room. The device runs with the shipped tuning table, as the benchmark's does.

Every output is what the entry point wrote: hits, occlusion bytes, images. Hits are single
precision in a fixed operation order and do not depend on the tree or the visiting order (ties go
to the smaller instance and primitive), so every correct version gives the same bits.
"""
import math

import numpy as np
import torch

import luisacompute_amd as lc
from luisacompute_amd import autotune, programs, workloads

EXTENT = 100.0
T_MAX = 1000.0          # beyond the scene's diagonal; finite, so that misses compare
FULL = 1 << 24          # triangles at which the soup's vertices spread by 0.5
_program = {}           # what a program makes once: device, stream, resident rooms, compiled kernels


# ------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # a small resident model and the smallest batch of the batched workload: picking, probes, one
        # tile of a preview; bound by the call and its launches
        dict(name="closest_model_4k", kind="closest", scene="sphere", tris=81920, rays=4096, view="camera"),
        # a scene of ordinary size, incoherent rays, odd counts: global illumination, simulation
        dict(name="closest_soup_1m", kind="closest", scene="soup", tris=1000003, rays=2097151, view="box"),
        # shadow rays of one light over a large scene
        dict(name="any_soup_4m", kind="any", scene="soup", tris=4194304, rays=4194301, view="light"),
        # the benchmark's step: 16.7M new triangles built for speed of build, 8.4M incoherent rays
        dict(name="frame_soup_16m_fast_build", kind="frame", scene="soup", tris=FULL, rays=1 << 23, view="box",
             hint="fast_build"),
        # a scene loaded and looked at once, with the options a program gets by default
        dict(name="frame_soup_1m_default", kind="frame", scene="soup", tris=1048577, rays=921600, view="camera",
             hint="fast_trace"),
        # a small mesh made anew for every frame: many launches over little work
        dict(name="frame_model_5k_default", kind="frame", scene="sphere", tris=5120, rays=16384, view="camera",
             hint="fast_trace"),
        # a deforming model, updated in place, seen by a 1080p camera
        dict(name="animate_model_1m", kind="animate", scene="sphere", tris=1000000, rays=2073600, view="camera"),
        # the instanced workload's 1,024 instances, 48 of them moved, 16 batches between 4,096 and 1M rays
        dict(name="instances_1024", kind="instances", instances=1024, moved=48, batches=16, largest=1 << 20),
        # the query benchmark's scene at half size: cutout triangles and spheres in AABBs
        dict(name="query_mixed", kind="query", tris=524288, boxes=524288, rays=2097152),
        # four samples per pixel of a 1080p view of the benchmark's room
        dict(name="render_room_1080p", kind="render", quads=512, width=1920, height=1080, spp=4, depth=8,
             form="wavefront"),
        # the run-time compiled path tracer on a preview of a smaller room
        dict(name="shader_room_preview", kind="shader", quads=128, width=640, height=360, spp=2, depth=8),
        # a burst of small and medium requests to a render server
        dict(name="serve_room_burst", kind="serve", quads=256, requests=12),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closest", "closest", "any", "frame", "frame", "animate", "instances", "query", "render",
                       "shader", "serve"])
    if kind in ("closest", "any", "frame", "animate"):
        c = dict(kind=kind, scene="sphere" if kind == "animate" else rng.choice(["soup", "soup", "sphere"]))
        c["tris"] = _log(rng, 320, 1 << 22 if kind == "animate" else (1 << 23 if kind == "closest" else FULL))
        c["rays"] = _log(rng, 1000, 1 << 22)
        c["view"] = "light" if kind == "any" else rng.choice(["box", "camera"])
        if kind == "frame":
            c["hint"] = rng.choice(["fast_trace", "fast_build"])
            if c["hint"] == "fast_trace":
                c["tris"] = min(c["tris"], _log(rng, 1 << 20, 1 << 22))
        return c
    if kind == "instances":
        n = _log(rng, 2, 4096)
        return dict(kind=kind, instances=n, moved=min(n, rng.randint(1, 64)), batches=rng.randint(1, 24),
                    largest=_log(rng, 8192, 1 << 20))
    if kind == "query":
        return dict(kind=kind, tris=_log(rng, 1000, 1 << 20), boxes=_log(rng, 1000, 1 << 20),
                    rays=_log(rng, 1000, 1 << 21))
    if kind == "render":
        return dict(kind=kind, quads=rng.choice([16, 64, 128, 256, 512]), width=rng.randint(64, 1920),
                    height=rng.randint(64, 1080), spp=rng.randint(1, 4), depth=rng.randint(2, 8),
                    form=rng.choice(["wavefront", "wavefront", "megakernel"]))
    if kind == "shader":
        return dict(kind=kind, quads=rng.choice([16, 64, 128, 256]), width=rng.randint(64, 1280),
                    height=rng.randint(64, 720), spp=rng.randint(1, 2), depth=rng.randint(2, 8))
    return dict(kind=kind, quads=rng.choice([16, 64, 128, 256]), requests=rng.randint(1, 24))


# ------------------------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _soup(n, g):
    """(3n, 4) vertices: centres uniform in the scene, vertices normal around them."""
    sigma = 0.5 * (FULL / n) ** (1.0 / 3.0)
    v = torch.zeros(n, 3, 4, device="cuda")
    v[..., :3] = torch.rand(n, 1, 3, generator=g, device="cuda") * EXTENT
    v[..., :3] += torch.randn(n, 3, 3, generator=g, device="cuda") * sigma
    return v.reshape(-1, 4), torch.arange(3 * n, device="cuda", dtype=torch.int32).reshape(-1, 3)


def _sphere(n, g):
    """A closed wavy sphere of at most n triangles (latitude rows of quads), waves from the seed."""
    rows = max(2, int(math.sqrt(n / 4.0)))
    cols = max(3, n // (2 * rows))
    i = torch.arange(rows + 1, device="cuda").reshape(-1, 1)
    j = torch.arange(cols, device="cuda").reshape(1, -1)
    theta, phi = i * (math.pi / rows), j * (2.0 * math.pi / cols)
    a = torch.rand(6, generator=g, device="cuda")
    r = 38.0 + 2.0 * torch.sin((3 + 4 * a[0]).floor() * phi + 6.28 * a[1]) * torch.sin(theta) ** 2 \
        + 2.0 * a[2] * torch.cos((2 + 5 * a[3]).floor() * theta + 6.28 * a[4])
    v = torch.zeros(rows + 1, cols, 4, device="cuda")
    v[..., 0] = 50.0 + r * torch.sin(theta) * torch.cos(phi)
    v[..., 1] = 50.0 + r * torch.cos(theta) + 0.0 * phi
    v[..., 2] = 50.0 + r * torch.sin(theta) * torch.sin(phi)
    i, j = i[:-1], j
    p00, p01 = i * cols + j, i * cols + (j + 1) % cols
    p10, p11 = p00 + cols, p01 + cols
    t = torch.stack([torch.stack([p00, p10, p11], -1), torch.stack([p00, p11, p01], -1)], 2)
    return v.reshape(-1, 4).contiguous(), t.reshape(-1, 3).to(torch.int32).contiguous()


def _directions(n, g):
    z = 1.0 - 2.0 * torch.rand(n, generator=g, device="cuda")
    phi = 2.0 * math.pi * torch.rand(n, generator=g, device="cuda")
    r = torch.sqrt(torch.clamp(1.0 - z * z, min=0.0))
    return torch.stack([r * torch.cos(phi), r * torch.sin(phi), z], 1)


def _rays(n, view, g, lo=0.0, hi=EXTENT):
    """(n, 8): origin, t_min, direction, t_max. box: uniform origins and directions; camera: pixels
    of a frame in raster order, jittered; light: segments from scene points to a point above it."""
    r = torch.zeros(n, 8, device="cuda")
    if view == "box":
        r[:, :3] = lo + (hi - lo) * torch.rand(n, 3, generator=g, device="cuda")
        r[:, 4:7] = _directions(n, g)
        r[:, 7] = T_MAX
    elif view == "camera":
        w = max(1, int(math.sqrt(n * 16.0 / 9.0)))
        h = -(-n // w)
        p = torch.arange(n, device="cuda")
        x = ((p % w) + torch.rand(n, generator=g, device="cuda")) / w - 0.5
        y = (torch.div(p, w, rounding_mode="floor") + torch.rand(n, generator=g, device="cuda")) / h - 0.5
        d = torch.stack([1.2 * x, -0.9 * y, torch.ones_like(x)], 1)
        r[:, :3] = torch.tensor([50.0, 52.0, -60.0], device="cuda")
        r[:, 4:7] = d / d.norm(dim=1, keepdim=True)
        r[:, 7] = T_MAX
    else:
        r[:, :3] = lo + (hi - lo) * torch.rand(n, 3, generator=g, device="cuda")
        to = torch.tensor([40.0, 160.0, 30.0], device="cuda") + 20.0 * torch.rand(n, 3, generator=g, device="cuda") - r[:, :3]
        far = to.norm(dim=1, keepdim=True)
        r[:, 4:7] = to / far
        r[:, 7] = 0.999 * far[:, 0]
    return r


def _geometry(case, g):
    return (_soup if case["scene"] == "soup" else _sphere)(case["tris"], g)


# ------------------------------------------------------------------------------------- the program
class _Memory:
    """A framework buffer as torch sees it (the buffer stays alive with the tensor)."""

    def __init__(self, buffer, shape, typestr):
        self.buffer = buffer
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(buffer.native, False), version=3,
                                             strides=None)


def _view(buffer, shape, typestr="<f4"):
    return torch.as_tensor(_Memory(buffer, shape, typestr), device="cuda")


def _device():
    if not _program:
        torch.cuda.init()
        dev = lc.Device(0)
        autotune.load_default(dev)
        _program.update(device=dev, stream=dev.create_stream(), rooms={}, kernel=None)
    return _program["device"], _program["stream"]


def _upload(dev, t, stride):
    """A framework buffer holding the tensor's values."""
    buf = dev.create_buffer(stride, max(1, t.numel() * t.element_size() // stride))
    _view(buf, tuple(t.shape), "<f4" if t.dtype == torch.float32 else "<i4").copy_(t)
    return buf


def _hits(dev, n):
    """A buffer of n hits and its fields."""
    buf = dev.create_buffer(24, n)
    f, i = _view(buf, (n, 6)), _view(buf, (n, 6), "<i4")
    f.zero_()
    return buf, dict(inst=i[:, 0], prim=i[:, 1], bary=f[:, 2:4], t=f[:, 4])


def _mesh(dev, v, t, hint="fast_trace", update=False):
    vb, tb = _upload(dev, v, 16), _upload(dev, t, 12)
    opt = lc.AccelOption(lc.AccelOption.FAST_TRACE if hint == "fast_trace" else lc.AccelOption.FAST_BUILD, 1,
                         1 if update else 0)
    return dev.create_mesh(vb, tb, option=opt)


def _room(quads):
    """The room's accel, materials and scene: resident, made once per size."""
    dev, stream = _device()
    if quads not in _program["rooms"]:
        room = workloads.BoxRoom(wall_quads=quads, block_quads=max(4, quads // 4))
        accel, _, inst = room.build(dev, stream)
        scene = room.scene()
        _program["rooms"][quads] = (accel, inst, scene, programs.PathTracerBindings(dev, stream, accel, inst, scene),
                                    room.triangle_count)
        stream.synchronize()
    return _program["rooms"][quads]


def _requests(case):
    """(width, height, spp) of the case's requests: the serving workload's mix, scaled to previews."""
    r = np.random.RandomState(case["requests"])
    return [(int(r.choice([64, 256, 512])), int(r.choice([64, 256, 512])), int(r.choice([1, 4, 16])))
            for _ in range(case["requests"])]


def prepare(case, seed):
    dev, stream = _device()
    g = _generator(seed)
    kind = case["kind"]
    s = dict(case=case, seed=int(seed))
    if kind in ("closest", "any", "frame", "animate"):
        v, t = _geometry(case, g)
        s["rays"] = _upload(dev, _rays(case["rays"], case["view"], g), 32)
        mesh = s["mesh"] = _mesh(dev, v, t, case.get("hint", "fast_trace"), kind == "animate")
        accel = s["accel"] = dev.create_accel()
        if kind == "animate":
            s["moved"] = _upload(dev, _sphere(case["tris"], g)[0], 16)
        if kind == "any":
            s["hits"] = dev.create_buffer(1, case["rays"])
            s["out"] = _view(s["hits"], (case["rays"],), "|u1")
        else:
            s["hits"], s["out"] = _hits(dev, case["rays"])
        torch.cuda.synchronize()
        if kind != "frame":
            stream << mesh.build()
        if kind in ("closest", "any"):
            accel.emplace_back(mesh)
            stream << accel.build()
        elif kind == "animate":
            accel.emplace_back(mesh)
    elif kind == "instances":
        meshes = s["meshes"] = [_mesh(dev, *_centred(*(_soup if k % 2 else _sphere)(n, g)))
                                for k, n in enumerate((1280, 5000, 20480, 60000, 81920, 200000, 327680, 500000))]
        n = case["instances"]
        s["affines"] = _affines(n, g)
        s["moves"] = _affines(case["moved"], g)
        s["moving"] = np.random.RandomState(seed).permutation(n)[:case["moved"]].tolist()
        accel = s["accel"] = dev.create_accel()
        torch.cuda.synchronize()
        for m in meshes:
            stream << m.build()
        for k in range(n):
            accel.emplace_back(meshes[k % 8], s["affines"][k])
        stream << accel.build()
        sizes = np.exp(np.random.RandomState(case["batches"]).uniform(np.log(4096), np.log(case["largest"]),
                                                                      case["batches"])).astype(int).tolist()
        s["batches"], s["out"] = [], []
        for k in sizes:
            hits = dev.create_buffer(24, k)
            s["batches"].append((_upload(dev, _rays(k, "box", g, -60.0, 60.0), 32), hits, k))
            s["out"].append((_view(hits, (k, 6), "<i4")[:, :2], _view(hits, (k, 6))[:, 2:5]))
    elif kind == "query":
        v, t = _soup(case["tris"], g)
        centre = torch.rand(case["boxes"], 3, generator=g, device="cuda") * EXTENT
        half = 0.5 * (FULL / case["boxes"]) ** (1.0 / 3.0) * (0.5 + torch.rand(case["boxes"], 3, generator=g, device="cuda"))
        s["mesh"] = _mesh(dev, v, t)
        s["prim"] = dev.create_procedural_primitive(_upload(dev, torch.cat([centre - half, centre + half], 1), 24))
        s["rays"] = _upload(dev, _rays(case["rays"], "box", g), 32)
        s["hits"] = dev.create_buffer(24, case["rays"])
        f, i = _view(s["hits"], (case["rays"], 6)), _view(s["hits"], (case["rays"], 6), "<i4")
        s["out"] = dict(inst=i[:, 0], prim=i[:, 1], bary=f[:, 2:4], hit_type=i[:, 4], t=f[:, 5])
        torch.cuda.synchronize()
        accel = s["accel"] = dev.create_accel()
        stream << s["mesh"].build() << s["prim"].build()
        accel.emplace_back(s["mesh"], opaque=False)
        accel.emplace_back(s["prim"])
        stream << accel.build()
    elif kind in ("render", "shader"):
        s["room"] = _room(case["quads"])
        w, h = case["width"], case["height"]
        s["image"] = dev.create_buffer(16, w * h)
        s["out"] = _view(s["image"], (h, w, 4))
        if kind == "render":
            o = s["options"] = lc.PtOptions()
            o.width, o.height, o.spp, o.max_depth, o.rr_depth = w, h, case["spp"], case["depth"], 3
            o.seed, o.sequence = s["seed"], 3 << 32
            o.mode = lc.PT_WAVEFRONT if case["form"] == "wavefront" else lc.PT_MEGAKERNEL
            chunk, o.sort, fetch = autotune.pathtracer_options(autotune.load_table())
            o.chunk_spp, o.graph, (o.fetch_chunk, o.fetch_segments) = chunk, 1, fetch
        elif _program["kernel"] is None:
            _program["kernel"] = programs.path_tracer.compile(dev)
    else:
        accel, inst, scene, _, _ = _room(case["quads"])
        server = s["server"] = lc.Server(dev, hbm_budget=64 << 20, wave_paths=4 << 20)
        s["scene"] = server.add_scene(accel, inst, scene)
        s["requests"] = [(w, h, spp, dev.create_buffer(16, w * h)) for w, h, spp in _requests(case)]
        s["out"] = [_view(b, (h, w, 4)) for w, h, _, b in s["requests"]]
    stream.synchronize()
    return s


def _centred(v, t):
    """The geometry scaled into [-1, 1]^3."""
    v[:, :3] = (v[:, :3] - 50.0) / 50.0
    return v, t


def _affines(n, g):
    """n rotations (uniform), scales U[0.5, 2] and translations U[-50, 50]^3 as 3x4 rows."""
    q = torch.randn(n, 4, generator=g, device="cuda", dtype=torch.float64)
    w, x, y, z = (q / q.norm(dim=1, keepdim=True)).unbind(1)
    m = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                     2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                     2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).reshape(n, 3, 3)
    m = m * (0.5 + 1.5 * torch.rand(n, 1, 1, generator=g, device="cuda", dtype=torch.float64))
    p = -50.0 + 100.0 * torch.rand(n, 3, 1, generator=g, device="cuda", dtype=torch.float64)
    return torch.cat([m, p], 2).cpu().numpy().astype(np.float32)


# ------------------------------------------------------------------------------------- one pass
def run(state):
    dev, stream = _device()
    case = state["case"]
    kind = case["kind"]
    if kind == "closest":
        state["accel"].trace_closest(stream, state["rays"], state["hits"], case["rays"])
    elif kind == "any":
        state["accel"].trace_any(stream, state["rays"], state["hits"], case["rays"])
    elif kind == "frame":
        accel, mesh = state["accel"], state["mesh"]
        stream << mesh.build(lc.BUILD_FORCE_BUILD)
        if len(accel) == 0:
            accel.emplace_back(mesh)
        else:
            accel.set(0, mesh)
        stream << accel.build()
        accel.trace_closest(stream, state["rays"], state["hits"], case["rays"])
    elif kind == "animate":
        accel, mesh = state["accel"], state["mesh"]
        stream << mesh.vb.copy_from_buffer(state["moved"]) << mesh.build()
        stream << accel.build()
        accel.trace_closest(stream, state["rays"], state["hits"], case["rays"])
    elif kind == "instances":
        accel = state["accel"]
        for k, m in zip(state["moving"], state["moves"]):
            accel.set_transform_on_update(k, m)
        stream << accel.build()
        accel.trace_batched(stream, state["batches"])
    elif kind == "query":
        state["accel"].query(stream, state["rays"], state["hits"], case["rays"], surface=lc.QUERY_SURFACE_CUTOUT,
                             cutout=0.8, procedural=lc.QUERY_PROCEDURAL_SPHERE)
    elif kind == "render":
        accel, inst, scene, _, _ = state["room"]
        accel.pathtrace(stream, inst, scene, state["options"], state["image"])
    elif kind == "shader":
        args = state["room"][3].args(state["image"], case["spp"], 0, case["depth"], 3, state["seed"], 3 << 32)
        stream << _program["kernel"](*args).dispatch(case["width"], case["height"])
    else:
        server = state["server"]
        for k, (w, h, spp, image) in enumerate(state["requests"]):
            server.submit(state["scene"], w, h, spp, image, seed=state["seed"], sequence=k << 32)
        server.drain()
    return state["out"]


# ------------------------------------------------------------------------------------- what it takes
def work(case):
    """Inputs read once, outputs written once; operations of a balanced 8-wide tree over the geometry
    (a box test of 8 children per level, two triangle tests) per ray."""
    kind = case["kind"]

    def per_ray(tris):
        return 8 * 12 * max(1.0, math.log(max(8, tris), 8)) + 2 * 50

    if kind in ("closest", "any", "frame", "animate"):
        n, r = case["tris"], case["rays"]
        out = 1 if kind == "any" else 24
        verts = 48 if case["scene"] == "soup" else 8
        return dict(bytes=n * (12 + verts) + r * (32 + out) + (2 * n * verts if kind == "animate" else 0),
                    flops=r * per_ray(n))
    if kind == "instances":
        sizes = np.exp(np.random.RandomState(case["batches"]).uniform(np.log(4096), np.log(case["largest"]),
                                                                      case["batches"])).astype(int)
        r = int(sizes.sum())
        return dict(bytes=1196360 * 40 + r * 56 + case["instances"] * 64, flops=r * per_ray(case["instances"]))
    if kind == "query":
        n, b, r = case["tris"], case["boxes"], case["rays"]
        return dict(bytes=n * 60 + b * 24 + r * 56, flops=r * per_ray(n + b))
    tris = 12 * case["quads"] ** 2 + 24 * max(4, case["quads"] // 4) ** 2
    if kind == "serve":
        paths = sum(w * h * spp for w, h, spp in _requests(case))
        pixels = sum(w * h for w, h, _ in _requests(case))
        depth = 8
    else:
        pixels = case["width"] * case["height"]
        paths = pixels * case["spp"]
        depth = case["depth"]
    # about half of the bounces live on, each with a closest and a shadow ray
    return dict(bytes=tris * 20 + pixels * 16, flops=paths * (1 + depth) * per_ray(tris))


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------------------------- in 64 bits
def _nearest(v, t, rays):
    """Nearest hit of each ray by testing every triangle in double precision."""
    p = v[:, :3].double()[t.long()]
    a, e1, e2 = p[:, 0], p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    n = torch.linalg.cross(e1, e2)
    o, d = rays[:, :3].double(), rays[:, 4:7].double()
    lo, hi = rays[:, 3].double(), rays[:, 7].double()
    out_t, out_b = hi.clone(), torch.zeros(len(rays), 2, dtype=torch.float64, device=v.device)
    step = max(1, (1 << 26) // max(1, len(t)))
    inf = torch.tensor(math.inf, dtype=torch.float64, device=v.device)
    # with s = o - a: t = -n.s / n.d, u = -(s x d).e2 / n.d, v = (s x d).e1 / n.d, as matrix products
    for k in range(0, len(rays), step):
        ok, dk = o[k:k + step], d[k:k + step]
        den = dk @ n.T
        tt = ((a * n).sum(1)[None] - ok @ n.T) / den
        od = torch.linalg.cross(ok, dk)
        ad2, ad1 = torch.linalg.cross(e2, a), torch.linalg.cross(e1, a)
        # (s x d).e = (o x d).e - (a x d).e, and (a x d).e = d.(e x a)
        u = -(od @ e2.T - dk @ ad2.T) / den
        w = (od @ e1.T - dk @ ad1.T) / den
        inside = (u >= 0) & (w >= 0) & (u + w <= 1) & (tt >= lo[k:k + step, None]) & (tt <= hi[k:k + step, None])
        tt = torch.where(inside, tt, inf)
        best, at = tt.min(1)
        hit = torch.isfinite(best)
        out_t[k:k + step] = torch.where(hit, best, hi[k:k + step])
        pick = torch.stack([u.gather(1, at[:, None])[:, 0], w.gather(1, at[:, None])[:, 0]], 1)
        out_b[k:k + step] = torch.where(hit[:, None], pick, torch.zeros_like(pick))
    return out_t, out_b


def exact(case, seed):
    """Distances and barycentrics by brute force, where the pairs of rays and triangles are few enough
    (whole numbers have no 64-bit value, path-traced images and queries no brute-force one in time)."""
    if case["kind"] not in ("closest", "frame", "animate") or case["tris"] * case["rays"] > 2 * 10 ** 9:
        return None
    g = _generator(seed)
    v, t = _geometry(case, g)
    rays = _rays(case["rays"], case["view"], g)
    if case["kind"] == "animate":
        v = _sphere(case["tris"], g)[0]
    out_t, out_b = _nearest(v, t, rays)
    return dict(inst=None, prim=None, bary=out_b, t=out_t)
