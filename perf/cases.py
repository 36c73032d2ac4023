"""The work that programs have this framework do, as cases that can be timed.

Every case goes through the public entry points of `radeonrays_sdk_amd.api`.
`listed()` names twelve of them, `draw(rng)` gives more of the same ranges.
`prepare(case, seed)` makes what a program holds before the call (geometry,
rays, built acceleration structures, result and scratch buffers, a captured
frame), `run(state)` makes one pass and returns its outputs whole, `work(case)`
says what a pass cannot do without and `exact(case, seed)` what it returns in
64-bit arithmetic.

Scenes are those of `radeonrays_sdk_amd.scenes` (triangle soups, fBm
heightfields, instanced soups, batches of small meshes, serving requests),
generated on the GPU from the seed.

Kinds and what they stand for:
  trace     one query on one geometry: picking and probes (1,000 rays),
            primary rays of an image, incoherent rays; "both" is a step that
            asks for the closest hit and for any hit of the same rays
  instanced secondary rays of an image of a two-level scene with large
            geometries (ambient occlusion or one diffuse bounce)
  serving   one batch of requests of very different sizes on several resident
            geometries, closest and any mixed
  build     a geometry built from triangles, with the default flags
            (restructured for tracing) or with PREFER_FAST_BUILD
  refit     a built geometry updated to moved vertices
  frame     a captured frame of a dynamic scene of many small meshes: all of
            them built (or refitted), then queried
  scene     a frame of moving instances: the top level built over them, then
            primary rays
  sort      the radix sort of (key, value) pairs by itself
"""
import math

import torch

from radeonrays_sdk_amd import api

HIT_BYTES = {"full": 16, "full_t": 32, "instance": 4}
NODE_BYTES = 64
HEADER_BYTES = 128
FAR = 100.0  # far end of every ray: past each single-level scene (unit cube) and inside float32's exact range

_context = None


def _ctx():
    """The program's one context, on torch's current stream."""
    global _context
    if _context is None:
        _context = api.Context(0)
    return _context


# --- cases -------------------------------------------------------------------


def listed():
    return [
        # The smallest serving request: a probe of 1,000 rays, latency alone.
        {"name": "probe_1k", "kind": "trace", "mesh": "soup", "tris": 65536, "default_build": True, "rays": 1000,
         "from": "sphere", "query": "closest", "output": "full"},
        # Primary rays of a 1024 x 1024 image of the 65,536-triangle soup.
        {"name": "camera_1m", "kind": "trace", "mesh": "soup", "tris": 65536, "default_build": True, "rays": 1 << 20,
         "from": "camera", "query": "closest", "output": "full_t"},
        # The benchmark's step: closest and any hits of 4M incoherent rays above a 1M-triangle terrain.
        {"name": "terrain_step_4m", "kind": "trace", "mesh": "terrain", "tris": 1045458, "default_build": True,
         "rays": 4 << 20, "from": "sphere", "query": "both", "output": "full"},
        # Two secondary rays per pixel of a 1024 x 1024 image: 64 soups of 10k-500k triangles, 4,096 instances.
        {"name": "instanced_2m", "kind": "instanced", "meshes": 64, "instances": 4096, "lo": 10000, "hi": 500000,
         "side": 1024},
        # One launch of the serving loop: 32 requests of 1k-1M rays over eight resident scenes.
        {"name": "serving_32", "kind": "serving", "scenes": 8, "lo": 10000, "hi": 1000000, "requests": 32,
         "max_rays": 1000000},
        # A small object built when it is loaded, 16-bit indices.
        {"name": "build_997", "kind": "build", "mesh": "soup", "tris": 997, "default_build": True, "index_bits": 16},
        # The terrain built for tracing (default flags).
        {"name": "build_1m", "kind": "build", "mesh": "terrain", "tris": 1045458, "default_build": True,
         "index_bits": 32},
        # A deforming object rebuilt on each frame (PREFER_FAST_BUILD).
        {"name": "build_fast_333k", "kind": "build", "mesh": "soup", "tris": 333333, "default_build": False,
         "index_bits": 32},
        # The terrain refitted to moved heights.
        {"name": "refit_1m", "kind": "refit", "mesh": "terrain", "tris": 1045458, "default_build": False},
        # 2,048 small meshes rebuilt and queried (256 any-hit rays each) by one captured frame.
        {"name": "frame_2048", "kind": "frame", "meshes": 2048, "lo": 64, "hi": 16384, "rays": 256, "op": "build",
         "query": "any"},
        # 1,000 moving instances of 16 props: the top level rebuilt, then 512 x 512 occlusion rays.
        {"name": "scene_1000", "kind": "scene", "meshes": 16, "tris": 2000, "instances": 1000, "side": 512,
         "query": "any", "output": "instance"},
        # 16M (Morton code, index) pairs.
        {"name": "sort_16m", "kind": "sort", "n": 1 << 24, "bits": 30},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("trace", "trace", "trace", "instanced", "serving", "build", "build", "refit", "frame", "scene",
                       "sort"))
    mesh = rng.choice(("soup", "terrain"))
    if kind == "trace":
        return {"kind": kind, "mesh": mesh, "tris": _log_int(rng, 1000, 1000000),
                "default_build": rng.random() < 0.7, "rays": _log_int(rng, 1000, 2 << 20),
                "from": rng.choice(("camera", "sphere")), "query": rng.choice(("closest", "closest", "any", "both")),
                "output": rng.choice(("full", "full", "full_t", "instance"))}
    if kind == "instanced":
        return {"kind": kind, "meshes": rng.randint(4, 48), "instances": _log_int(rng, 64, 4096), "lo": 5000,
                "hi": _log_int(rng, 20000, 300000), "side": rng.randint(200, 900)}
    if kind == "serving":
        return {"kind": kind, "scenes": rng.randint(2, 8), "lo": 10000, "hi": _log_int(rng, 50000, 1000000),
                "requests": rng.randint(4, 32), "max_rays": _log_int(rng, 20000, 500000)}
    if kind == "build":
        tris = _log_int(rng, 100, 1000000)
        return {"kind": kind, "mesh": mesh, "tris": tris, "default_build": rng.random() < 0.5,
                "index_bits": 16 if tris <= 20000 and rng.random() < 0.5 else 32}
    if kind == "refit":
        return {"kind": kind, "mesh": mesh, "tris": _log_int(rng, 1000, 1000000), "default_build": rng.random() < 0.5}
    if kind == "frame":
        return {"kind": kind, "meshes": _log_int(rng, 32, 1500), "lo": 64, "hi": _log_int(rng, 1000, 16384),
                "rays": rng.randint(60, 256), "op": rng.choice(("build", "refit")),
                "query": rng.choice(("closest", "any"))}
    if kind == "scene":
        return {"kind": kind, "meshes": rng.randint(4, 32), "tris": _log_int(rng, 200, 5000),
                "instances": _log_int(rng, 50, 2000), "side": rng.randint(100, 512),
                "query": rng.choice(("closest", "any")), "output": rng.choice(("full", "instance"))}
    return {"kind": kind, "n": _log_int(rng, 4000, 12000000), "bits": rng.choice((30, 30, 32))}


# --- scenes, on the GPU ------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda")


def _soup(tris, g):
    """Centroids uniform in the unit cube, corners N(0, 0.01^2) around them."""
    c = _rand(g, tris, 1, 3)
    v = c + 0.01 * torch.randn(tris, 3, 3, generator=g, device="cuda")
    return v.reshape(-1, 3), torch.arange(3 * tris, dtype=torch.int32, device="cuda").reshape(-1, 3)


def _heights(res, g, octaves=6):
    """fBm value noise on a res x res grid: random lattices, smoothstep between them, rescaled to [0, 0.2]."""
    x = torch.linspace(0.0, 1.0, res, device="cuda")
    total = torch.zeros(res, res, device="cuda")
    for o in range(octaves):
        cells = 4 << o
        lattice = _rand(g, cells + 2, cells + 2)
        f = x * cells
        i = f.floor().long()
        t = f - i
        s = t * t * (3.0 - 2.0 * t)
        rows = lattice[i] * (1.0 - s)[:, None] + lattice[i + 1] * s[:, None]
        total += 0.5 ** o * (rows[:, i] * (1.0 - s) + rows[:, i + 1] * s)
    return 0.2 * (total - total.min()) / (total.max() - total.min()).clamp_min(1e-12)


def _terrain(tris, g):
    """A heightfield over the unit square with about `tris` triangles, two per cell."""
    res = max(2, int(round(math.sqrt(tris / 2.0))) + 1)
    x = torch.linspace(0.0, 1.0, res, device="cuda")
    v = torch.stack([x.expand(res, res), _heights(res, g), x[:, None].expand(res, res)], dim=-1).reshape(-1, 3)
    a = (torch.arange(res - 1, device="cuda")[:, None] * res + torch.arange(res - 1, device="cuda")).reshape(-1)
    b, c, d = a + 1, a + res, a + res + 1
    tri = torch.stack([a, b, c, b, d, c], dim=1).reshape(-1, 3)
    return v.contiguous(), tri.to(torch.int32)


def _mesh(kind, tris, g):
    return _soup(tris, g) if kind == "soup" else _terrain(tris, g)


def _tri_count(kind, tris):
    return tris if kind == "soup" else 2 * max(1, int(round(math.sqrt(tris / 2.0)))) ** 2


def _rays(origins, directions, far=FAR):
    r = torch.zeros(origins.shape[0], 8, device="cuda")
    r[:, 0:3] = origins
    r[:, 4:7] = directions
    r[:, 7] = far
    return r


def _sphere(n, g):
    return torch.nn.functional.normalize(torch.randn(n, 3, generator=g, device="cuda"), dim=1)


def _camera(n, eye, g, far=FAR):
    """n primary rays in scan-line order of a 45 degree camera looking along +z, jittered within their pixels."""
    w = max(1, math.isqrt(n))
    h = -(-n // w)
    k = torch.arange(n, device="cuda")
    j = _rand(g, n, 2)
    t = math.tan(math.radians(22.5))
    px = ((k % w) + j[:, 0]) / w * 2 - 1
    py = 1 - ((k // w) + j[:, 1]) / h * 2
    d = torch.nn.functional.normalize(torch.stack([px * t, py * t, torch.ones_like(px)], dim=1), dim=1)
    return _rays(torch.tensor(eye, device="cuda").expand(n, 3), d, far)


def _mesh_rays(mesh, n, how, g):
    if how == "camera":
        return _camera(n, (0.5, 0.5, -1.5) if mesh == "soup" else (0.5, 0.35, -0.2), g)
    o = _rand(g, n, 3)
    if mesh == "terrain":
        o[:, 1] = 0.25 + 0.25 * o[:, 1]
    return _rays(o, _sphere(n, g))


def _transforms(n, g, trans):
    """Uniform rotations, scales in [0.5, 2], translations in [-trans, trans]^3: [n, 3, 4] on the host."""
    q = torch.nn.functional.normalize(torch.randn(n, 4, generator=g, device="cuda"), dim=1)
    x, y, z, w = q.unbind(1)
    rot = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                       2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                       2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], dim=1).reshape(n, 3, 3)
    rot = rot * (0.5 + 1.5 * _rand(g, n, 1, 1))
    move = trans * (2.0 * _rand(g, n, 3, 1) - 1.0)
    return torch.cat([rot, move], dim=2).cpu().numpy()


def _log_sizes(n, lo, hi, g):
    """n sizes spread evenly over the logarithm of [lo, hi], in an order of the seed's."""
    sizes = [int(lo * (hi / lo) ** ((k + 0.5) / n)) for k in range(n)]
    return [sizes[k] for k in torch.randperm(n, generator=g, device="cuda").tolist()]


def _built(ctx, meshes, default_build):
    """The meshes' geometries, their results in one allocation."""
    sizes = [ctx.geometry_requirements(int(i.shape[0]), int(v.shape[0]), default_build).result_buffer_size
             for v, i in meshes]
    return [ctx.build_geometry(v, i, restructure=default_build, result=r)
            for (v, i), r in zip(meshes, ctx.result_arena(sizes))]


# --- states ------------------------------------------------------------------


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, _ctx(), _gen(seed))


def _prepare_trace(case, ctx, g):
    v, i = _mesh(case["mesh"], case["tris"], g)
    rays = _mesh_rays(case["mesh"], case["rays"], case["from"], g)
    accel = ctx.build_geometry(v, i, restructure=case["default_build"])
    queries = ("closest", "any") if case["query"] == "both" else (case["query"],)
    hits = {q: ctx.empty(case["rays"] * HIT_BYTES[case["output"]]) for q in queries}
    return {"kind": "trace", "ctx": ctx, "accel": accel, "rays": rays, "output": case["output"], "hits": hits,
            "scratch": ctx.trace_scratch(case["rays"])}


def _prepare_instanced(case, ctx, g):
    """The secondary rays of a primary pass: cosine-distributed about the hit triangle's normal, two per pixel, the
    pixels in scan-line order; a pixel that saw nothing has rays with an empty interval."""
    sizes = _log_sizes(case["meshes"], case["lo"], case["hi"], g)
    meshes = [_soup(n, g) for n in sizes]
    blases = _built(ctx, meshes, True)
    trans = 50.0 * (case["instances"] / 4096.0) ** (1.0 / 3.0)
    pick = torch.randint(0, len(meshes), (case["instances"],), generator=g, device="cuda")
    xf = _transforms(case["instances"], g, trans)
    scene = ctx.build_scene([blases[k] for k in pick.tolist()], xf)
    n = case["side"] ** 2
    primary = _camera(n, (0.0, 0.0, -3.0 * trans), g, far=1e30)
    hit = ctx.intersect(scene, primary, "closest", "full_t").view(torch.int32).view(-1, 8)
    inst = hit[:, 2].long()
    seen = inst >= 0
    inst = inst.clamp_min(0)
    t = hit.view(torch.float32)[:, 4]
    first = torch.tensor([0] + sizes, device="cuda").cumsum(0)  # first triangle of each mesh
    corners = torch.cat([m[0].reshape(-1, 3, 3) for m in meshes])
    tri = corners[(first[pick[inst]] + hit[:, 3].long().clamp_min(0)).clamp_max(corners.shape[0] - 1)]
    m = torch.from_numpy(xf).cuda()[inst][:, :, :3]
    e = tri[:, 1:] - tri[:, :1]
    normal = torch.linalg.cross((m * e[:, None, 0]).sum(2), (m * e[:, None, 1]).sum(2))
    normal = torch.nn.functional.normalize(normal, dim=1)
    normal = torch.where((normal * primary[:, 4:7]).sum(1, keepdim=True) > 0, -normal, normal)
    p = primary[:, 0:3] + t[:, None] * primary[:, 4:7]
    p = p + 1e-4 * (1.0 + p.abs().amax(1, keepdim=True)) * normal
    up = torch.nn.functional.normalize(normal[:, None] + 0.999 * _sphere(2 * n, g).view(n, 2, 3), dim=2)
    rays = torch.zeros(n, 2, 8, device="cuda")
    rays[:, :, 0:3] = torch.where(seen[:, None], p, torch.zeros_like(p))[:, None]
    rays[:, :, 4:7] = torch.where(seen[:, None, None], up, torch.tensor([0.0, 0.0, 1.0], device="cuda"))
    rays[:, :, 7] = torch.where(seen, 1e30, -1.0)[:, None]
    rays = rays.view(-1, 8)
    return {"kind": "trace", "ctx": ctx, "accel": scene, "rays": rays, "output": "full",
            "hits": {"closest": ctx.empty(2 * n * 16)}, "scratch": ctx.trace_scratch(2 * n)}


def _prepare_serving(case, ctx, g):
    """Requests as the serving loop coalesces them: log-uniform ray counts, each a slice of a camera or a sphere pool of
    its scene's kind, 70 % closest hit."""
    kinds = ["soup" if k % 2 == 0 else "terrain" for k in range(case["scenes"])]
    sizes = _log_sizes(case["scenes"], case["lo"], case["hi"], g)
    blases = _built(ctx, [_mesh(k, n, g) for k, n in zip(kinds, sizes)], True)
    pools = {(m, how): _mesh_rays(m, case["max_rays"], how, g) for m in ("soup", "terrain") for how in ("camera", "sphere")}
    counts = _log_sizes(case["requests"], 1000, case["max_rays"], g)
    scene = torch.randint(0, case["scenes"], (case["requests"],), generator=g, device="cuda").tolist()
    u = _rand(g, case["requests"], 3).tolist()
    total = sum(-(-n // 16) * 16 for n in counts)
    hits = torch.zeros(total * 16, dtype=torch.uint8, device="cuda")  # each request's hits on a 256-byte boundary
    requests, at = [], 0
    for n, k, (a, b, c) in zip(counts, scene, u):
        pool = pools[kinds[k], "camera" if a < 0.5 else "sphere"]
        off = int(b * (pool.shape[0] - n))
        requests.append((blases[k], pool[off:off + n], "closest" if c < 0.7 else "any", "full", hits[16 * at:16 * (at + n)]))
        at += -(-n // 16) * 16
    return {"kind": "serving", "ctx": ctx, "requests": requests, "hits": hits,
            "scratch": ctx.batch_scratch(len(requests), sum(counts), max(counts))}


def _prepare_build(case, ctx, g):
    v, i = _mesh(case["mesh"], case["tris"], g)
    if case["index_bits"] == 16:
        i = i.to(torch.int16)  # the bits of unsigned 16-bit indices
    req = ctx.geometry_requirements(int(i.shape[0]), int(v.shape[0]), case["default_build"])
    return {"kind": "build", "ctx": ctx, "mesh": (v, i), "default_build": case["default_build"],
            "result": ctx.empty(req.result_buffer_size), "scratch": ctx.empty(req.temporary_build_buffer_size)}


def _prepare_refit(case, ctx, g):
    v, i = _mesh(case["mesh"], case["tris"], g)
    accel = ctx.build_geometry(v, i, restructure=case["default_build"])
    moved = v.clone()
    moved[:, 1] += 1e-3 * torch.randn(v.shape[0], generator=g, device="cuda")
    return {"kind": "refit", "ctx": ctx, "accel": accel, "mesh": (moved, i)}


def _prepare_frame(case, ctx, g):
    sizes = _log_sizes(case["meshes"], case["lo"], case["hi"], g)
    v, i = _soup(sum(sizes), g)
    at = [0]
    for n in sizes:
        at.append(at[-1] + n)
    meshes = [(v[3 * a:3 * (a + n)], i[:n]) for a, n in zip(at, sizes)]
    per = case["rays"]
    rays = _rays(_rand(g, len(sizes) * per, 3), _sphere(len(sizes) * per, g))
    results = ctx.result_arena([ctx.geometry_requirements(n, 3 * n).result_buffer_size for n in sizes])
    scratch = ctx.empty(ctx.batch_build_requirements(meshes))
    accels = ctx.build_geometry_batch(meshes, scratch=scratch, results=results)
    hits = torch.zeros(rays.shape[0] * 16, dtype=torch.uint8, device="cuda")
    requests = [(a, rays[k * per:(k + 1) * per], case["query"], "full", hits[16 * k * per:16 * (k + 1) * per])
                for k, a in enumerate(accels)]
    qscratch = ctx.batch_scratch(len(requests), rays.shape[0], per)
    if case["op"] == "refit":
        moved = v + 1e-3 * torch.randn(v.shape, generator=g, device="cuda")
        meshes = [(moved[3 * a:3 * (a + n)], i[:n]) for a, n in zip(at, sizes)]
    # One frame, captured as an engine's render loop does: its host work is recorded once.
    torch.cuda.synchronize()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side, capture_error_mode="relaxed"):
        with ctx.on_stream(side):
            if case["op"] == "refit":
                ctx.update_geometry_batch(accels, meshes, scratch=scratch)
            else:
                ctx.build_geometry_batch(meshes, scratch=scratch, results=results)
            ctx.intersect_batch(requests, scratch=qscratch)
    torch.cuda.synchronize()
    return {"kind": "frame", "graph": graph, "hits": hits, "keep": (meshes, requests, scratch, qscratch)}


def _prepare_scene(case, ctx, g):
    blases = _built(ctx, [_soup(case["tris"], g) for _ in range(case["meshes"])], True)
    trans = 10.0
    pick = torch.randint(0, case["meshes"], (case["instances"],), generator=g, device="cuda").tolist()
    xf = _transforms(case["instances"], g, trans)
    n = case["side"] ** 2
    rays = _camera(n, (0.0, 0.0, -3.0 * trans), g, far=1e30)
    return {"kind": "scene", "ctx": ctx, "blases": [blases[k] for k in pick], "transforms": xf, "rays": rays,
            "output": case["output"], "query": case["query"], "hits": ctx.empty(n * HIT_BYTES[case["output"]]),
            "scratch": ctx.trace_scratch(n)}


def _prepare_sort(case, ctx, g):
    n, top = case["n"], 1 << case["bits"]
    keys = torch.randint(0, top, (n,), generator=g, device="cuda", dtype=torch.int64)
    pairs = torch.stack([keys.to(torch.int32), torch.arange(n, dtype=torch.int32, device="cuda")])
    return {"kind": "sort", "ctx": ctx, "pairs": pairs, "work": pairs.clone(), "bits": case["bits"],
            "tmp": (torch.empty_like(pairs[0]), torch.empty_like(pairs[0])), "scratch": ctx.empty(_sort_bytes(ctx, n))}


def _sort_bytes(ctx, n):
    from ctypes import byref, c_size_t

    from radeonrays_sdk_amd import rr
    size = c_size_t()
    rr.check(ctx.lib.rrxGetSortMemoryRequirements(ctx.ctx, n, byref(size)), "rrxGetSortMemoryRequirements")
    return size.value


# --- one pass ----------------------------------------------------------------


def run(state):
    return globals()["_run_" + state["kind"]](state)


def _fields(hits, output):
    """A hit buffer's fields, as views of it."""
    if output == "instance":
        return {"ids": hits.view(torch.int32)}
    f, w = hits.view(torch.float32), hits.view(torch.int32)
    if output == "full":
        return {"uv": f.view(-1, 4)[:, :2], "ids": w.view(-1, 4)[:, 2:]}
    return {"uv": f.view(-1, 8)[:, :2], "ids": w.view(-1, 8)[:, 2:4], "t": f.view(-1, 8)[:, 4]}


def _run_trace(s):
    return {q: _fields(s["ctx"].intersect(s["accel"], s["rays"], q, s["output"], hits=h, scratch=s["scratch"]), s["output"])
            for q, h in s["hits"].items()}


def _run_serving(s):
    s["ctx"].intersect_batch(s["requests"], scratch=s["scratch"])
    return _fields(s["hits"], "full")


def _nodes(accel):
    """The node array that follows the header, as 64-byte records."""
    n = 2 * accel.prim_count - 1
    return accel.buffer[HEADER_BYTES:HEADER_BYTES + n * NODE_BYTES].view(torch.int32).view(n, NODE_BYTES // 4)


def _run_build(s):
    v, i = s["mesh"]
    return _nodes(s["ctx"].build_geometry(v, i, restructure=s["default_build"], scratch=s["scratch"], result=s["result"]))


def _run_refit(s):
    s["ctx"].update_geometry(s["accel"], *s["mesh"])
    return _nodes(s["accel"])


def _run_frame(s):
    s["graph"].replay()
    return _fields(s["hits"], "full")


def _run_scene(s):
    scene = s["ctx"].build_scene(s["blases"], s["transforms"])
    hits = s["ctx"].intersect(scene, s["rays"], s["query"], s["output"], hits=s["hits"], scratch=s["scratch"])
    return _fields(hits, s["output"])


def _run_sort(s):
    # The sort is in place: the pairs of this pass come from the program's own.
    s["work"].copy_(s["pairs"])
    s["ctx"].sort_pairs(s["work"][0], s["work"][1], key_bits=s["bits"], tmp=s["tmp"], scratch=s["scratch"])
    return s["work"]


# --- what a pass cannot do without -------------------------------------------


def _depth(tris):
    return math.log2(max(2, tris))


def _query_work(rays, tris, node_total, hit_bytes, queries=1):
    """Rays read and hits written once, and the nodes on each ray's path or all of them once, whichever is less;
    12 operations per box and 60 per triangle test, a path of log2(triangles) nodes."""
    d = _depth(tris)
    nodes = min(node_total * NODE_BYTES, rays * d * NODE_BYTES)
    return {"bytes": queries * (rays * (32 + hit_bytes) + nodes), "flops": queries * rays * (24 * d + 60)}


def _build_work(tris, vertices, index_bytes=4, topology=True):
    """Vertices and indices read once, nodes written once (a refit also reads their links)."""
    nodes = (2 * tris - 1) * NODE_BYTES
    return {"bytes": vertices * 12 + tris * 3 * index_bytes + nodes + (0 if topology else (2 * tris - 1) * 12),
            "flops": tris * 30}


def _add(*ws):
    return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}


def _mean_log(lo, hi):
    return (hi - lo) / math.log(hi / lo) if hi > lo else lo


def work(case):
    kind = case["kind"]
    if kind == "trace":
        n = _tri_count(case["mesh"], case["tris"])
        return _query_work(case["rays"], n, 2 * n - 1, HIT_BYTES[case["output"]], 2 if case["query"] == "both" else 1)
    if kind == "instanced":
        tris = _mean_log(case["lo"], case["hi"])
        nodes = 2 * (case["meshes"] * tris + case["instances"])
        return _query_work(2 * case["side"] ** 2, tris * case["instances"], nodes, 16)
    if kind == "serving":
        tris = _mean_log(case["lo"], case["hi"])
        return _query_work(case["requests"] * _mean_log(1000, case["max_rays"]), tris, 2 * tris * case["scenes"], 16)
    if kind in ("build", "refit"):
        n = _tri_count(case["mesh"], case["tris"])
        vertices = 3 * n if case["mesh"] == "soup" else (int(math.isqrt(n // 2)) + 1) ** 2
        return _build_work(n, vertices, case.get("index_bits", 32) // 8, kind == "build")
    if kind == "frame":
        tris = _mean_log(case["lo"], case["hi"])
        total = case["meshes"] * tris
        return _add(_build_work(total, 3 * total, 4, case["op"] == "build"),
                    _query_work(case["meshes"] * case["rays"], tris, 2 * total, 16))
    if kind == "scene":
        n = case["instances"]
        build = {"bytes": n * (56 + 96 + 2 * NODE_BYTES), "flops": n * 400}
        return _add(build, _query_work(case["side"] ** 2, n * case["tris"], 2 * (n + case["meshes"] * case["tris"]),
                                       HIT_BYTES[case["output"]]))
    return {"bytes": 16.0 * case["n"], "flops": 1.0 * case["n"]}  # keys and values read once and written once


# --- the same in 64 bits -----------------------------------------------------


def exact(case, seed):
    """Barycentrics (and distances) of closest hits by brute force over all triangles, where that is a short
    computation; sorted pairs by torch's stable sort.  Nodes are the inputs' own numbers: nothing is computed."""
    g = _gen(seed)
    if case["kind"] == "sort":
        n = case["n"]
        keys = torch.randint(0, 1 << case["bits"], (n,), generator=g, device="cuda", dtype=torch.int64)
        keys, order = torch.sort(keys, stable=True)
        return torch.stack([keys.to(torch.int32), order.to(torch.int32)])
    if case["kind"] != "trace" or case["query"] != "closest" or case["output"] == "instance":
        return None
    if case["mesh"] != "soup" or case["rays"] * case["tris"] > 2e9:
        return None  # terrain rays may cross shared edges, where two triangles share the hit
    v, _ = _soup(case["tris"], g)
    rays = _mesh_rays(case["mesh"], case["rays"], case["from"], g).double()
    tri = v.double().view(-1, 3, 3)
    v0, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    uv = torch.zeros(case["rays"], 2, dtype=torch.float64, device="cuda")
    ts = rays[:, 7].clone()
    step = max(1, int(2e7 // case["tris"]))
    for a in range(0, case["rays"], step):
        o, d = rays[a:a + step, None, 0:3], rays[a:a + step, None, 4:7]
        p = torch.linalg.cross(d.expand(-1, e2.shape[0], -1), e2[None].expand(d.shape[0], -1, -1))
        det = (p * e1).sum(2)
        s = o - v0
        u = (s * p).sum(2) / det
        q = torch.linalg.cross(s, e1[None].expand(s.shape[0], -1, -1))
        w = (q * d).sum(2) / det
        t = (q * e2).sum(2) / det
        inside = (u >= 0) & (w >= 0) & (u + w <= 1) & (t >= 0) & (t <= FAR)
        best, k = torch.where(inside, t, math.inf).min(1)
        hit = best < math.inf
        pick = torch.stack([u.gather(1, k[:, None])[:, 0], w.gather(1, k[:, None])[:, 0]], dim=1)
        uv[a:a + step] = torch.where(hit[:, None], pick, uv[a:a + step])
        ts[a:a + step] = torch.where(hit, best, ts[a:a + step])
    out = {"uv": uv, "ids": None}
    return {"closest": {**out, "t": ts} if case["output"] == "full_t" else out}
