"""The framework's measured cases: what a program that uses it has it do.

Each case is one pass through the public entry points of
`mambatracer_amd.api`, over inputs made from a seed.  Kinds:

  render    one render job (`api.render`, or a captured `api.RenderGraph`)
  adaptive  the first frames after a camera move, the light grid learning
  batch     many uneven jobs through the shared queues (`api.Batch`)
  rays      closest hit, shadow rays and any hit over a batch of rays
  records   closest hit and compaction on the reference's own records
  compact   stable compaction of a path queue
  surface   BSDF, environment and light-grid sampling over a batch of hits
  bvh       the device BVH builder

Every result of the framework is defined bit for bit (the same IEEE
operations in the same order whatever the kernels look like), so every
case's tolerance is "exact".
"""
import math

import numpy as np
import torch

from mambatracer_amd import _lib, api
from mambatracer_amd import workloads as W

_context = []


def _ctx():
    """A program's one context (one device, one queue), kept for its life."""
    if not _context:
        _context.append(api.Context(0))
    return _context[0]


# --------------------------------------------------------------------- cases
def listed():
    return [
        # an interactive preview while the user moves the camera: one sample
        # per pixel of a small window, then the tone-mapped ARGB frame;
        # launches and latency are what counts
        {"name": "preview", "kind": "render", "scene": "soup", "size": 20000, "width": 160, "height": 90, "spp": 1,
         "light": "env", "captured": False, "tail": 0, "show": True},
        # a room lit by its own emitting triangles (no environment), as the
        # default scene of the reference is
        {"name": "room_lights", "kind": "render", "scene": "room", "size": 20000, "width": 512, "height": 512,
         "spp": 4, "light": "mesh", "captured": False, "tail": 0, "show": False},
        # a serving-sized job on a dense soup; odd image, odd sample count
        {"name": "job_soup", "kind": "render", "scene": "soup", "size": 150001, "width": 317, "height": 241,
         "spp": 13, "light": "env", "captured": False, "tail": 0, "show": False},
        # the headline frame: 1M triangles, 1080p, 16 samples, the environment
        # sampled through the light grid, replayed from its captured render
        {"name": "frame_1080p", "kind": "render", "scene": "spheres", "size": 256, "width": 1920, "height": 1080,
         "spp": 16, "light": "guided", "captured": True, "tail": 3, "show": False},
        # two frames after a camera move: grid reseeded, rendered, updated,
        # rendered again with what it learned, and shown
        {"name": "adaptive_540p", "kind": "adaptive", "size": 64, "width": 960, "height": 540, "spp": 2},
        # serving: uneven jobs of resident scenes through the shared queues
        {"name": "batch_24", "kind": "batch", "jobs": 24, "scenes": 6, "side_hi": 400, "spp_hi": 24},
        # the stress batch: 64M random rays through 4M triangles, sorted by
        # origin first (the mode the autotuner picks for such batches)
        {"name": "rays_random_64m", "kind": "rays", "scene": "cluster", "size": 4000000, "rays": 64 << 20,
         "camera": False, "mode": _lib.MT_TRACE_PACKED_BINNED},
        # visibility queries of one camera image, default mode, odd size
        {"name": "rays_camera_1m", "kind": "rays", "scene": "room", "size": 20000, "rays": 1021 * 1021,
         "camera": True, "mode": 0},
        # the drop-in path: 80-byte rays and 96-byte hit records in place
        {"name": "records_512k", "kind": "records", "size": 20000, "rays": 733 * 719},
        # a 1080p x 16 queue of which 45% lives on: id, origin, direction
        {"name": "compact_33m", "kind": "compact", "items": 1920 * 1080 * 16, "live": 0.45, "widths": "4,16,16"},
        # the shading stages one call at a time over a batch of hits
        {"name": "surface_2m", "kind": "surface", "items": 2000003},
        # a mesh rebuilt on the device after an edit
        {"name": "bvh_1m", "kind": "bvh", "scene": "spheres", "size": 1048578},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["render", "render", "render", "adaptive", "batch", "rays", "rays", "records", "compact",
                       "surface", "bvh"])
    if kind == "render":
        scene = rng.choice(["soup", "room", "spheres"])
        size = {"soup": (1000, 500000), "room": (1000, 200000), "spheres": (4, 256)}[scene]
        light = "mesh" if scene == "room" else rng.choice(["env", "guided", "both" if scene == "soup" else "env"])
        # soups scatter every path inside the cloud: their jobs are the sizes
        # of the multi-job workload; the open sphere scene goes to 1080p
        w = _log_int(rng, 64, 1920 if scene == "spheres" else 900)
        h = max(48, min(1080, int(w * rng.uniform(0.5, 1.0))))
        most = 33_000_000 if scene == "spheres" else 4_000_000
        spp = max(1, min(_log_int(rng, 1, 33) - 1 or 1, most // (w * h)))
        return {"kind": kind, "scene": scene, "size": _log_int(rng, *size), "width": w, "height": h, "spp": spp,
                "light": light, "captured": rng.random() < 0.3, "tail": rng.choice([0, 0, 0, 3]),
                "show": rng.random() < 0.3}
    if kind == "adaptive":
        w = _log_int(rng, 128, 1920)
        return {"kind": kind, "size": _log_int(rng, 4, 128), "width": w, "height": int(w * rng.uniform(0.5, 0.75)),
                "spp": rng.randint(1, 4)}
    if kind == "batch":
        return {"kind": kind, "jobs": rng.randint(4, 40), "scenes": rng.randint(2, 8),
                "side_hi": _log_int(rng, 100, 500), "spp_hi": rng.randint(4, 32)}
    if kind == "rays":
        if rng.random() < 0.5:
            side = _log_int(rng, 64, 2000)
            return {"kind": kind, "scene": rng.choice(["room", "soup"]), "size": _log_int(rng, 1000, 500000),
                    "rays": side * side, "camera": True, "mode": 0}
        return {"kind": kind, "scene": rng.choice(["cluster", "soup"]), "size": _log_int(rng, 1000, 2000000),
                "rays": _log_int(rng, 10000, 30_000_000), "camera": False,
                "mode": rng.choice([0, _lib.MT_TRACE_PACKED_BINNED, _lib.MT_TRACE_PACKED_POOL])}
    if kind == "records":
        side = _log_int(rng, 64, 1500)
        return {"kind": kind, "size": _log_int(rng, 1000, 300000), "rays": side * side}
    if kind == "compact":
        return {"kind": kind, "items": _log_int(rng, 10000, 33_000_000), "live": round(rng.uniform(0.02, 0.98), 3),
                "widths": rng.choice(["4,16,16", "8,16,16,16", "16,16", "4", "4,8"])}
    if kind == "surface":
        return {"kind": kind, "items": _log_int(rng, 10000, 12_000_000)}
    return {"kind": kind, "scene": rng.choice(["spheres", "soup", "cluster"]),
            "size": _log_int(rng, 5000, 2_000_000)}


# ------------------------------------------------------------------- inputs
def _mesh(scene, size, seed):
    """(points, faces, normals or None) of about `size` triangles
    (`spheres`: of `size` spheres)."""
    seed = int(seed) & 0xFFFFF
    if scene == "spheres":
        p, n, f = api.gen_spheres(seed, size)
        return p, f, n
    if scene == "cluster":  # nine in ten tiny and close together, the rest large and far apart
        tiny = size * 9 // 10
        p0, f0 = api.gen_soup(seed, tiny, -0.05, 0.05, 1e-4, 1e-3)
        p1, f1 = api.gen_soup(seed + 1000, size - tiny, -100.0, 100.0, 1.0, 10.0, first_vertex=p0.shape[0])
        return np.concatenate([p0, p1]), np.concatenate([f0, f1]), None
    if scene == "room":
        p0, f0 = api.gen_room(0)
        p1, f1 = api.gen_soup(seed, size, -0.8, 0.8, 0.01, 0.05, first_vertex=8)
        return np.concatenate([p0, p1]), np.concatenate([f0, f1]), None
    p, f = api.gen_soup(seed, size, -0.8, 0.8, 0.01, 0.05)
    return p, f, None


def _scene(scene, size, seed, emit=False, materials=257):
    """The scene on the device, its triangles' materials drawn uniformly
    (spheres carry their own); emit: one triangle in 200 is a light."""
    p, f, n = _mesh(scene, size, seed)
    if scene != "spheres":
        r = np.random.default_rng(int(seed))
        f[:, 9] = r.integers(0, materials, f.shape[0])
        if emit:
            f[::200, 9] = materials
    nodes, bounds, depth = api.CNormalBVH.build(p, f)
    return api.Scene(_ctx(), p, f, nodes, bounds, depth, normals=n), bounds


def _materials(seed):
    """257 surfaces, then one emitter."""
    m = W.c1_materials(seed=int(seed) & 0xFFFFF)
    return np.concatenate([m, W.material_records(np.full((1, 3), 0.5), 0.04, 0.5, 0.5,
                                                 emission=np.full((1, 3), 1.0), emission_power=20.0)])


def _environment(seed):
    r = np.random.default_rng(int(seed) + 17)
    env = api.CEnvironment(_ctx())
    env.setEnvironmentMap(W.env_map(sun_u=float(r.uniform(0.1, 0.9)), sun_v=float(r.uniform(0.1, 0.45))))
    return env


def _grid(env, pos):
    grid = api.CAdaptiveEnvironment(_ctx())
    tile = api.lightgrid_seed_tile(env.lum.cpu().numpy(), env.w, env.h)
    grid.setHDRLuminance(tile)
    grid.setCameraPosition(pos)
    env.attachLightGrid(grid)
    return grid, tile


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _unit(n, g):
    v = torch.randn((n, 4), generator=g, device="cuda")
    v[:, 3] = 0
    return (v / v[:, :3].norm(dim=1, keepdim=True)).contiguous()


def _job(case, seed):
    if case["scene"] == "spheres":
        return W.RenderJob(width=case["width"], height=case["height"], spp=case["spp"], seed=seed & 0x7FFFFFFF)
    j = W.soup_job(W.JobSpec(0, 0, 8, case["spp"], seed & 0x7FFFFFFF))
    j.width, j.height = case["width"], case["height"]
    return j


def prepare(case, seed):
    ctx = _ctx()
    return {"ctx": ctx, "case": case, **_PREPARE[case["kind"]](ctx, case, int(seed))}


def _prepare_render(ctx, case, seed):
    light = case["light"]
    scene, _ = _scene(case["scene"], case["size"], seed, emit=light in ("mesh", "both"))
    mats = ctx.to_device(_materials(seed))
    job = _job(case, seed)
    job.flags = _lib.MT_RENDER_TAIL_FROM(case["tail"])
    env = None if light == "mesh" else _environment(seed)
    lf = nl = None
    if light in ("mesh", "both"):
        lf, nl = api.mesh_lights(ctx, scene, mats)
        job.flags |= _lib.MT_RENDER_PICKED_LIGHT
    if light == "guided":  # as the render thread leaves the grid: seeded, one frame, one update
        grid, _ = _grid(env, job.pos)
        job.flags |= _lib.MT_RENDER_LIGHTGRID_ENV
        api.render(ctx, scene, mats, env, job, stats=False)
        grid.update()
    s = {"scene": scene, "mats": mats, "env": env, "job": job, "lf": lf, "nl": nl}
    if case["captured"]:
        s["graph"] = api.RenderGraph(ctx, scene, mats, env, job, light_faces=lf, num_lights=nl)
    if case["show"]:
        s["view"] = api.CImage(ctx, job.width, job.height)
    return s


def _prepare_adaptive(ctx, case, seed):
    scene, _ = _scene("spheres", case["size"], seed)
    env = _environment(seed)
    job = _job({**case, "scene": "spheres"}, seed)
    job.flags = _lib.MT_RENDER_LIGHTGRID_ENV
    grid, tile = _grid(env, job.pos)
    return {"scene": scene, "mats": ctx.to_device(_materials(seed)), "env": env, "job": job, "grid": grid,
            "tile": tile, "view": api.CImage(ctx, job.width, job.height)}


def _prepare_batch(ctx, case, seed):
    # the jobs' sizes belong to the case; their scenes and random numbers to the seed
    r = np.random.default_rng([case["jobs"], case["scenes"], case["side_hi"], case["spp_hi"]])
    size = [int(math.exp(r.uniform(math.log(1000), math.log(100000)))) for _ in range(case["scenes"])]
    scenes = [_scene("soup", n, seed + 1 + i)[0] for i, n in enumerate(size)]
    jobs = []
    for i in range(case["jobs"]):
        side = int(round(math.exp(r.uniform(math.log(64), math.log(case["side_hi"])))))
        spp = int(r.integers(1, case["spp_hi"] + 1))
        k = int(r.integers(0, len(scenes)))
        jobs.append((k, W.soup_job(W.JobSpec(i, k, side, spp, (seed * 1000 + i) & 0x7FFFFFFF))))
    engine = api.Batch(ctx, queue_capacity=1 << 21, arena_bytes=2 << 30, max_jobs=64,
                       policy=_lib.MT_BATCH_SMALLEST_FIRST)
    engine.set_iterations(8)
    return {"scenes": scenes, "mats": ctx.to_device(_materials(seed)), "env": _environment(seed), "jobs": jobs,
            "engine": engine}


def _camera_rays(n, seed):
    side = int(math.isqrt(n))
    r = np.random.default_rng(seed)
    return api.gen_camera_rays([float(r.uniform(-0.1, 0.1)), float(r.uniform(-0.1, 0.1)), -0.95], [0, 0, 1],
                               [0, 1, 0], 60.0, side, n // side)


def _prepare_rays(ctx, case, seed):
    scene, bounds = _scene(case["scene"], case["size"], seed)
    n = case["rays"]
    g = _gen(seed)
    lo = torch.tensor(bounds[0, :3], device="cuda")
    hi = torch.tensor(bounds[0, 4:7], device="cuda")
    if case["camera"]:
        o, d = (ctx.to_device(x) for x in _camera_rays(n, seed))
        light = np.array([0.3, 0.9, -0.2], np.float32)
    else:
        o = torch.empty((n, 4), device="cuda")
        o[:, :3] = lo + (hi - lo) * torch.rand((n, 3), generator=g, device="cuda")
        o[:, 3] = 0.001
        d = _unit(n, g)
        d[:, 3] = math.inf
        light = W.c2_light(bounds, seed=seed)
    return {"scene": scene, "o": o, "d": d, "light": light}


def _prepare_records(ctx, case, seed):
    scene, _ = _scene("soup", case["size"], seed)
    o, d = _camera_rays(case["rays"], seed)
    n = o.shape[0]
    fresh = ctx.to_device(api.ray_records(o, d))
    queue = torch.randperm(n, generator=_gen(seed), device="cuda").to(torch.int32)
    isects = torch.zeros((n, api.INTERSECTION_RECORD_WORDS), device="cuda")
    pixels = queue.clone()
    total = ctx.scalar_i32(0)
    compact = api.CCompact()
    compact.init(ctx, isects, pixels, total)
    return {"scene": scene, "fresh": fresh, "rays": fresh.clone(), "isects": isects, "queue": queue,
            "pixels": pixels, "total": total, "compact": compact}


def _prepare_compact(ctx, case, seed):
    g = _gen(seed)
    n = case["items"]
    live = round(case["live"] * n)
    flags = torch.zeros((n,), dtype=torch.int32, device="cuda")
    flags[torch.randperm(n, generator=g, device="cuda")[:live]] = 1
    pay = []
    for w in (int(x) // 4 for x in case["widths"].split(",")):
        x = torch.randint(-(1 << 31), (1 << 31) - 1, (n, w), generator=g, device="cuda", dtype=torch.int32)
        pay.append(x.reshape(n) if w == 1 else x)
    return {"flags": flags, "pay": pay, "length": ctx.scalar_i32(n), "live": live}


def _prepare_surface(ctx, case, seed):
    n = case["items"]
    g = _gen(seed)
    env = _environment(seed)
    grid, _ = _grid(env, W.RenderJob().pos)
    d = _unit(n, g)
    nrm = _unit(n, g)
    nrm = torch.where((nrm[:, :3] * d[:, :3]).sum(1, keepdim=True) > 0, -nrm, nrm).contiguous()
    mat = torch.randint(-1, 257, (n,), generator=g, device="cuda", dtype=torch.int32)  # -1: a miss
    hit = torch.rand((n, 4), generator=g, device="cuda") * 10 - 5
    hit[:, 3] = 0
    return {"env": env, "grid": grid, "mats": ctx.to_device(_materials(seed)), "d": d, "n": nrm, "mat": mat,
            "u3": torch.rand((n, 3), generator=g, device="cuda"), "u4": torch.rand((n, 4), generator=g, device="cuda"),
            "u2": torch.rand((n, 2), generator=g, device="cuda"), "hit": hit.contiguous(),
            "wi": _unit(n, g)[:, :3].contiguous(), "out": _unit(n, g)}


def _prepare_bvh(ctx, case, seed):
    size = max(1, case["size"] // 4096) if case["scene"] == "spheres" else case["size"]
    p, f, _ = _mesh(case["scene"], size, seed)
    return {"points": ctx.to_device(p), "faces": ctx.to_device(f)}


_PREPARE = {"render": _prepare_render, "adaptive": _prepare_adaptive, "batch": _prepare_batch, "rays": _prepare_rays,
            "records": _prepare_records, "compact": _prepare_compact, "surface": _prepare_surface,
            "bvh": _prepare_bvh}


# --------------------------------------------------------------------- pass
def run(state):
    return _RUN[state["case"]["kind"]](state["ctx"], state)


def _show(view, image):
    view.cFrameAccum.copy_(image)
    view.processImage()
    return view.getFrameARGB()


def _run_render(ctx, s):
    if "graph" in s:
        s["graph"].launch(s["job"].seed)
        image = s["graph"].image
    else:
        image, _ = api.render(ctx, s["scene"], s["mats"], s["env"], s["job"], light_faces=s["lf"],
                              num_lights=s["nl"], stats=False)
    return {"image": image, "argb": _show(s["view"], image)} if "view" in s else {"image": image}


def _run_adaptive(ctx, s):
    grid = s["grid"]
    grid.setHDRLuminance(s["tile"])  # the camera moved: the grid starts over
    first, _ = api.render(ctx, s["scene"], s["mats"], s["env"], s["job"], stats=False)
    grid.update()
    second, st = api.render(ctx, s["scene"], s["mats"], s["env"], s["job"])
    return {"first": first, "second": second, "argb": _show(s["view"], second),
            "rays": [int(st.extension_rays), int(st.shadow_rays)]}


def _run_batch(ctx, s):
    engine, images = s["engine"], []
    for tag, (k, job) in enumerate(s["jobs"]):
        images.append(ctx.empty((job.width * job.height, 4), torch.float32))
        engine.submit(tag, s["scenes"][k], s["mats"], s["env"], job, images[-1])
    engine.run()
    return images


def _run_rays(ctx, s):
    mode = s["case"]["mode"]
    prim, t, _ = api.intersect_primitives(ctx, s["scene"], s["o"], s["d"], mode=mode)
    so, sd, valid = api.shadow_rays(ctx, s["o"], s["d"], prim, t, s["light"])
    occ, _ = api.intersect_occlusion(ctx, s["scene"], so, sd, mode=mode)
    return {"prim": prim, "t": t, "valid": valid, "occluded": occ}


def _run_records(ctx, s):
    s["rays"].copy_(s["fresh"])      # the caller's camera fills its rays and its pixel queue
    s["pixels"].copy_(s["queue"])
    api.intersect_records(ctx, s["scene"], s["rays"], s["isects"])
    s["compact"].execute()
    return {"rays": s["rays"], "isects": s["isects"].view(torch.int32), "pixels": s["pixels"], "total": s["total"]}


def _run_compact(ctx, s):
    idx, count, out = api.compact(ctx, s["flags"], length=s["length"], payloads=s["pay"])
    n = s["live"]  # compaction writes the first `live` entries
    return {"index": idx[:n], "count": count, "out": [x[:n] for x in out]}


def _run_surface(ctx, s):
    rec, mid = api.bsdf_setup(ctx, s["d"], s["n"], s["n"], s["mat"], s["mats"])
    f, wi, pdf, cs = api.bsdf_sample(ctx, rec, mid, s["mats"], s["u3"])
    ef, epdf, ecs = api.bsdf_eval(ctx, rec, mid, s["mats"], s["wi"])
    env, grid = s["env"], s["grid"]
    return {"setup": (rec, mid), "sample": (f, wi, pdf, cs), "eval": (ef, epdf, ecs),
            "light": env.illuminate(s["u2"]), "radiance": env.radiance(s["out"]),
            "guided_light": env.illuminate_adaptive(grid, s["hit"], s["u4"]),
            "guided_radiance": env.radiance_adaptive(grid, s["out"], s["hit"], accumulate=False)}


def _run_bvh(ctx, s):
    nodes, bounds, depth = api.CNormalBVH.build_device(ctx, s["points"], s["faces"])
    return {"nodes": nodes, "bounds": bounds, "depth": depth}


_RUN = {"render": _run_render, "adaptive": _run_adaptive, "batch": _run_batch, "rays": _run_rays,
        "records": _run_records, "compact": _run_compact, "surface": _run_surface, "bvh": _run_bvh}


# --------------------------------------------------------------------- work
_BOX_PAIR, _TRIANGLE = 42, 50  # operations of one node's two box tests, of one triangle test


def _triangles(case):
    if case["kind"] == "bvh":
        return case["size"]
    return 4096 * case["size"] + 2 if case.get("scene", "spheres") == "spheres" else case["size"]


def _ray_flops(tris):
    """A ray's walk from the root to one leaf of a balanced tree."""
    return _BOX_PAIR * math.log2(max(2, tris)) + _TRIANGLE


def work(case):
    kind = case["kind"]
    if kind in ("render", "adaptive"):
        tris, px = _triangles(case), case["width"] * case["height"]
        frames = 2 if kind == "adaptive" else 1
        # one closest-hit and one shadow ray per path at the least; about 500
        # operations to shade a vertex
        return {"bytes": tris * (64 + 48) + frames * px * 16 + 1024 * 512 * 16,
                "flops": frames * px * case["spp"] * (2 * _ray_flops(tris) + 500)}
    if kind == "batch":
        side = (case["side_hi"] - 64) / math.log(case["side_hi"] / 64)  # mean of a log-uniform side
        px = case["jobs"] * side * (case["side_hi"] + 64) / 2
        return {"bytes": px * 16, "flops": px * (case["spp_hi"] + 1) / 2 * (2 * _ray_flops(10000) + 500)}
    if kind == "rays":
        n, tris = case["rays"], case["size"]
        return {"bytes": n * (32 + 8 + 4 + 4) + tris * (64 + 48), "flops": n * 2 * _ray_flops(tris)}
    if kind == "records":
        n = case["rays"]
        return {"bytes": n * (80 + 80 + 96 + 4 + 4), "flops": n * _ray_flops(case["size"])}
    if kind == "compact":
        b = sum(int(x) for x in case["widths"].split(","))
        return {"bytes": case["items"] * (4 + case["live"] * (2 * b + 4)), "flops": 0}
    if kind == "surface":
        # inputs once (d, n, mat, u3, u2, u4, hit, wi, out), outputs once
        n = case["items"]
        return {"bytes": n * (16 + 16 + 4 + 12 + 8 + 16 + 16 + 12 + 16
                              + 84 + 32 + 20 + 40 + 24 + 44 + 28), "flops": n * 1200}
    tris = case["size"]
    return {"bytes": tris * (3 * 16 + 40 + 2 * (28 + 32)), "flops": tris * 12 * math.log2(max(2, tris))}


def tolerance(case):
    return "exact"


# -------------------------------------------------------------------- exact
def exact(case, seed):
    """Plain torch in 64 bits.  Renders, batches and tree builds have none:
    a path's branches (which triangle, which lobe, whether it goes on) turn
    on single roundings, and a 64-bit path tracer in torch takes minutes."""
    kind = case["kind"]
    if kind == "compact":
        s = prepare(case, seed)
        keep = s["flags"].nonzero().reshape(-1)
        return {"index": keep.to(torch.int32), "count": torch.tensor([keep.numel()], dtype=torch.int32),
                "out": [x[keep] for x in s["pay"]]}
    if kind == "surface":
        return _exact_surface(prepare(case, seed))
    if kind in ("rays", "records") and case["rays"] * case["size"] <= 3e10:
        p, f, _ = _mesh(case["scene"] if kind == "rays" else "soup", case["size"], seed)
        if kind == "rays":
            if not case["camera"]:
                s = prepare(case, seed)
                t = _nearest(p, f, s["o"], s["d"])
            else:
                o, d = _camera_rays(case["rays"], seed)
                t = _nearest(p, f, torch.from_numpy(o).cuda(), torch.from_numpy(d).cuda())
            return {"prim": None, "t": t, "valid": None, "occluded": None}
        o, d = _camera_rays(case["rays"], seed)
        rays = torch.from_numpy(api.ray_records(o, d)).double()
        rays[:, 19] = _nearest(p, f, torch.from_numpy(o).cuda(), torch.from_numpy(d).cuda()).cpu()
        return {"rays": rays, "isects": None, "pixels": None, "total": None}
    return None


def _nearest(points, faces, o, d):
    """Distance to the nearest triangle of every ray (tMax where none), by
    testing every triangle."""
    v = torch.from_numpy(points).cuda().double()[:, :3]
    f = torch.from_numpy(faces).cuda().long()
    a = v[f[:, 0]]
    e1, e2 = v[f[:, 1]] - a, v[f[:, 2]] - a
    nrm = torch.linalg.cross(e1, e2)
    best = []
    step = max(1, int(3e8 // max(1, f.shape[0])))
    for i in range(0, o.shape[0], step):
        ro, rd = o[i:i + step].double(), d[i:i + step].double()
        # Moeller-Trumbore as scalar triple products, one matrix product each
        det = -rd[:, :3] @ nrm.T
        m = torch.linalg.cross(ro[:, :3], rd[:, :3])
        t = (ro[:, :3] @ nrm.T - (a * nrm).sum(1)) / det
        b1 = (rd[:, :3] @ torch.linalg.cross(a, e2).T + m @ e2.T) / det
        b2 = -(rd[:, :3] @ torch.linalg.cross(a, e1).T + m @ e1.T) / det
        ok = (b1 >= 0) & (b2 >= 0) & (b1 + b2 <= 1) & (t > ro[:, 3:4])
        t = torch.where(ok, t, torch.full_like(t, math.inf)).min(1).values
        best.append(torch.minimum(t, rd[:, 3]))
    return torch.cat(best)


def _dot(a, b):
    return (a * b).sum(-1)


def _ggx(mat, wi, wo, wh):
    """(value of the lobe without its tint, Schlick's fifth power, pdf as the
    framework states it: the generated direction is the view of the pdf)."""
    ax, ay = mat[:, 17], mat[:, 18]

    def lam(w):
        t2 = (ax * w[:, 0]) ** 2 + (ay * w[:, 1]) ** 2
        return (torch.sqrt(1 + t2 / w[:, 2] ** 2) - 1) / 2

    dist = 1 / (math.pi * ax * ay * ((wh[:, 0] / ax) ** 2 + (wh[:, 1] / ay) ** 2 + wh[:, 2] ** 2) ** 2)
    value = dist / (1 + lam(wi) + lam(wo)) / (4 * wi[:, 2].abs() * wo[:, 2].abs())
    c = _dot(wo, wh)
    pdf = dist / (1 + lam(wo)) * c.clamp(min=0.001) / wo[:, 2].clamp(min=0.001) / (4 * c)
    return value, (1 - c.abs()) ** 5, pdf


def _exact_surface(s):
    """setup and eval from the formulas; the sampled directions and the
    lights come of discrete picks (a lobe, a texel), so no value is stated."""
    n, d = s["n"].double()[:, :3], s["d"].double()[:, :3]
    a = 1 / (1 + n[:, 2])
    b = -n[:, 0] * n[:, 1] * a
    mx = torch.stack([1 - n[:, 0] ** 2 * a, b, -n[:, 0]], 1)
    my = torch.stack([b, 1 - n[:, 1] ** 2 * a, -n[:, 1]], 1)
    frame = torch.stack([mx, my, n], 1)
    fix = -(frame * d[:, None]).sum(2)
    geom = (frame * n[:, None]).sum(2)
    hit = (s["mat"] >= 0) & (fix[:, 2].abs() >= 1e-6)
    m = s["mats"].double()[s["mat"].clamp(min=0).long()]
    lum = torch.tensor([0.2989, 0.5866, 0.1145], dtype=torch.float64, device=m.device)
    ad, ag = _dot(m[:, 4:7] * m[:, 8:9], lum), _dot(m[:, 12:15] * m[:, 16:17], lum)
    rec = torch.zeros((n.shape[0], 20), dtype=torch.float64, device=n.device)
    rec[:, :9] = frame.reshape(-1, 9)
    rec[:, 9:12] = fix
    rec[:, 12:15] = torch.where(hit[:, None], geom, 0.0)
    rec[:, 15] = torch.where(hit, ad / (ad + ag), 0.0)
    rec[:, 16] = torch.where(hit, ag / (ad + ag), 0.0)
    gen = (frame * s["wi"].double()[:, None]).sum(2)
    same = gen[:, 2] * fix[:, 2] >= 0
    on = same & hit & (fix[:, 2] >= 1e-6) & (gen[:, 2] >= 1e-6)
    wh = fix + gen
    wh = wh / wh.norm(dim=1, keepdim=True)
    value, fifth, gpdf = _ggx(m, fix, gen, wh)
    f0 = m[:, 12:15]
    f = m[:, 4:7] / math.pi + (f0 + (1 - f0) * fifth[:, None]) * value[:, None]
    pdf = rec[:, 15] * gen[:, 2] / math.pi + rec[:, 16] * gpdf
    return {"setup": (rec, None), "sample": (None, None, None, None),
            "eval": (torch.where(on[:, None], f, 0.0), torch.where(on, pdf, 0.0), torch.where(same, gen[:, 2], 0.0)),
            "light": (None,) * 4, "radiance": (None,) * 3, "guided_light": (None,) * 5,
            "guided_radiance": (None,) * 4}
