"""Workloads of the ray-traversal engine, as a user's program runs them.

Each case is one call (or one burst of calls) of the public entry points on
device-resident rays: single traces of a few hundred to tens of millions of
rays, closest and any hit, CWBVH and BVH2, the reference's bind-and-trace entry
points, ambient occlusion straight from surfels, a captured multi-scene batch,
a served burst and a scene larger than the last-level cache.

Ray intervals, offsets and scene generators are those of cwbvh_amd.workloads:
a heightfield under ambient-occlusion rays, a lattice of spheres seen by a
1920x1080 camera, and a clustered triangle soup with unbounded diffuse rays.
"""
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import cwbvh_amd as cw
from cwbvh_amd import workloads as W

MODES = {"closest": cw.TRACE_CLOSEST, "any": cw.TRACE_ANY}

# Node visits and triangle tests per ray (CWBVH; BVH2 visits 2.8 times as many
# nodes of two children) that the path needs on each scene family.
VISITS = {"heightfield": (8.0, 4.5), "spheres": (7.0, 2.0), "soup": (20.0, 14.0)}


def listed():
    return [
        # a picking or probe query: one small launch, latency and launch cost count
        {"name": "query_small", "path": "trace", "kind": "cwbvh", "mesh": "heightfield", "triangles": 65536,
         "rays": 1000, "mode": "closest"},
        # ambient occlusion of a small lightmap: below the size of a persistent grid, ragged
        {"name": "occlusion_medium", "path": "trace", "kind": "cwbvh", "mesh": "spheres", "triangles": 300000,
         "rays": 393217, "mode": "any"},
        # the smallest of the named workloads: a million AO rays on a heightfield
        {"name": "ao_heightfield", "path": "trace", "kind": "cwbvh", "mesh": "heightfield", "triangles": 65536,
         "rays": 1048576, "mode": "closest"},
        # coherent camera rays with the triangle's index reported
        {"name": "camera", "path": "camera", "width": 1920, "height": 1080, "mode": "closest"},
        # a full AO frame, 16 rays per primary hit: the headline workload, both modes
        {"name": "frame_closest", "path": "frame", "kind": "cwbvh", "width": 1920, "height": 1080, "spp": 16,
         "mode": "closest"},
        {"name": "frame_any", "path": "frame", "kind": "cwbvh", "width": 1920, "height": 1080, "spp": 16,
         "mode": "any"},
        # the same scene through the binary BVH, the engine's second path
        {"name": "frame_bvh2", "path": "frame", "kind": "bvh2", "width": 1920, "height": 1080, "spp": 4,
         "mode": "closest"},
        # the reference's entry points on caller-owned arrays (80 B nodes): bind, trace, wait
        {"name": "bound_arrays", "path": "bound", "mesh": "spheres", "triangles": 980000, "rays": 4000037},
        # lightmap baking from surfels: rays made in the kernel, one occlusion count per surfel
        {"name": "surfel_bake", "path": "surfels", "mesh": "spheres", "triangles": 980000, "surfels": 260007,
         "spp": 32, "mode": "any"},
        # many scenes of very uneven size in one captured launch
        {"name": "scene_batch", "path": "batch", "scenes": 40, "max_triangles": 300000, "max_rays": 1000000,
         "mode": "closest"},
        # a scene that does not fit the last-level cache, incoherent rays, the scene's default configuration
        {"name": "large_soup", "path": "trace", "kind": "cwbvh", "mesh": "soup", "triangles": 5000000,
         "rays": 16777216, "mode": "closest"},
        # a burst of requests against resident scenes, results in place
        {"name": "served_burst", "path": "server", "scenes": 8, "max_triangles": 300000, "requests": 96,
         "max_rays": 131072, "mode": "closest"},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    mode = rng.choice(("closest", "any"))
    path = rng.choice(("trace", "trace", "trace", "frame", "frame", "camera", "bound", "surfels", "batch", "server",
                       "soup"))
    if path == "trace":
        return {"path": "trace", "kind": rng.choice(("cwbvh", "cwbvh", "bvh2")),
                "mesh": rng.choice(("heightfield", "spheres")), "triangles": size(2000, 1000000),
                "rays": size(300, 12000000), "mode": mode}
    if path == "soup":
        return {"path": "trace", "kind": "cwbvh", "mesh": "soup", "triangles": size(4800000, 5000000),
                "rays": size(300000, 16000000), "mode": mode}
    if path == "frame":
        return {"path": "frame", "kind": rng.choice(("cwbvh", "cwbvh", "bvh2")), "width": size(320, 1920),
                "height": size(200, 1080), "spp": rng.choice((1, 2, 4, 7)), "mode": mode}
    if path == "camera":
        return {"path": "camera", "width": size(320, 1920), "height": size(200, 1080), "mode": mode}
    if path == "bound":
        return {"path": "bound", "mesh": rng.choice(("heightfield", "spheres")), "triangles": size(2000, 980000),
                "rays": size(300, 4000037)}
    if path == "surfels":
        return {"path": "surfels", "mesh": rng.choice(("heightfield", "spheres")), "triangles": size(2000, 980000),
                "surfels": size(300, 260007), "spp": rng.choice((8, 16, 32)), "mode": mode}
    if path == "batch":
        return {"path": "batch", "scenes": size(3, 40), "max_triangles": size(20000, 300000),
                "max_rays": size(20000, 1000000), "mode": mode}
    return {"path": "server", "scenes": size(2, 8), "max_triangles": size(20000, 300000), "requests": size(8, 96),
            "max_rays": size(8192, 131072), "mode": mode}


# ------------------------------------------------------------------ inputs


def _mesh(kind, triangles, seed):
    if kind == "heightfield":
        return W.heightfield_of(triangles, seed)
    if kind == "spheres":
        return W.icospheres_of(triangles, seed)
    return W.c3_mesh(triangles, seed)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _corners(mesh):
    v = torch.from_numpy(mesh.vertices).cuda()
    f = torch.from_numpy(mesh.indices).cuda().long()
    return v[f[:, 0]], v[f[:, 1]], v[f[:, 2]]


def _surface(mesh, n, g, in_order=False):
    """n area-uniform points of the surface and their unit normals."""
    a, b, c = _corners(mesh)
    normal = torch.linalg.cross(b - a, c - a)
    area = normal.norm(dim=1).double()
    cum = torch.cumsum(area, 0)
    at = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * cum[-1]
    if in_order:
        at = at.sort().values
    tri = torch.searchsorted(cum, at).clamp_(max=len(cum) - 1)
    u = torch.rand(n, 2, generator=g, device="cuda")
    s = u[:, :1].sqrt()
    p = a[tri] * (1 - s) + b[tri] * (s * (1 - u[:, 1:])) + c[tri] * (s * u[:, 1:])
    nrm = normal[tri]
    return p, nrm / nrm.norm(dim=1, keepdim=True).clamp_min(1e-30)


def _hemisphere(nrm, g):
    """Cosine-weighted directions around unit normals."""
    d = torch.randn(nrm.shape, generator=g, device="cuda")
    d = nrm + d / d.norm(dim=1, keepdim=True).clamp_min(1e-12) * 0.9999
    return d / d.norm(dim=1, keepdim=True)


def _rays(o, d, tmax):
    r = torch.empty((len(o), 8), device="cuda")
    r[:, 0:3], r[:, 3], r[:, 4:7], r[:, 7] = o, 0.0, d, tmax
    return r


def _ao_rays(mesh, n, g, per_point=8):
    """Ambient-occlusion rays: area-uniform points with per_point rays each."""
    diag = mesh.diagonal()
    p, nrm = _surface(mesh, -(-n // per_point), g)
    p, nrm = p.repeat_interleave(per_point, 0)[:n], nrm.repeat_interleave(per_point, 0)[:n]
    return _rays(p + nrm * (1e-4 * diag), _hemisphere(nrm, g), 0.1 * diag)


def _diffuse_rays(mesh, n, g):
    """Secondary rays without bound: uniform directions from the surface."""
    p, nrm = _surface(mesh, n, g)
    d = torch.randn((n, 3), generator=g, device="cuda")
    d = d / d.norm(dim=1, keepdim=True).clamp_min(1e-12)
    side = (d * nrm).sum(1, keepdim=True).sign()
    return _rays(p + nrm * side * (1e-4 * mesh.diagonal()), d, math.inf)


def _layout(mesh, kind="cwbvh", threads=0):
    params = cw.default_build_params(num_threads=threads)
    bvh2, cwbvh = cw.build_layouts(mesh, params, bvh2=kind == "bvh2", cwbvh=kind == "cwbvh")
    return bvh2 if kind == "bvh2" else cwbvh


def _trace_state(scene, rays, flags):
    return {"scene": scene, "rays": rays, "hits": torch.empty((len(rays), 4), device="cuda"), "flags": flags}


def _camera_rays(case):
    c = W.C1_CAMERA
    return torch.from_numpy(cw.rays_pinhole(case["width"], case["height"], c["eye"], c["target"], c["up"], c["fov"],
                                            0.0, 1e30)).cuda()


def _frame_rays(case, mesh, g):
    """AO rays of a camera image: spp cosine rays per primary hit, pixel order."""
    prim = _camera_rays(case)
    hits = torch.empty((len(prim), 4), device="cuda")
    primary = cw.Scene(_layout(mesh))
    primary.trace(prim.data_ptr(), hits.data_ptr(), len(prim), cw.TRACE_CLOSEST | cw.TRACE_PRIM_ID)
    torch.cuda.synchronize()
    ids = hits.view(torch.int32)[:, 1].long()
    hit = ids >= 0
    a, b, c = _corners(mesh)
    ids, d = ids[hit], prim[hit, 4:7]
    nrm = torch.linalg.cross(b[ids] - a[ids], c[ids] - a[ids])
    nrm = nrm / nrm.norm(dim=1, keepdim=True).clamp_min(1e-30)
    nrm = torch.where((nrm * d).sum(1, keepdim=True) > 0, -nrm, nrm)
    diag = mesh.diagonal()
    o = prim[hit, 0:3] + d * hits[hit, 0:1] + nrm * (1e-4 * diag)
    nrm = nrm.repeat_interleave(case["spp"], 0)
    return _rays(o.repeat_interleave(case["spp"], 0), _hemisphere(nrm, g), 0.05 * diag)


def _plan(case, seed):
    """Scene sizes of a batch or a server: log-uniform, alternating families.
    Sizes and ray counts belong to the case, vertices and rays to the seed."""
    rng = np.random.default_rng([case["scenes"], case["max_triangles"], case["max_rays"]])
    lo, hi = math.log(1000), math.log(case["max_triangles"])
    return [("heightfield" if i % 2 == 0 else "spheres", int(math.exp(rng.uniform(lo, hi))), int(seed) * 1009 + i)
            for i in range(case["scenes"])], rng


def _scenes(plan):
    def make(entry):
        mesh = _mesh(*entry)
        return mesh, _layout(mesh, threads=2)

    with ThreadPoolExecutor(6) as ex:
        return [(mesh, cw.Scene(layout)) for mesh, layout in ex.map(make, plan)]


def prepare(case, seed):
    g = _generator(seed)
    flags = MODES[case.get("mode", "closest")]
    path = case["path"]
    if path == "trace":
        mesh = _mesh(case["mesh"], case["triangles"], seed)
        rays = (_diffuse_rays if case["mesh"] == "soup" else _ao_rays)(mesh, case["rays"], g)
        state = _trace_state(cw.Scene(_layout(mesh, case["kind"])), rays, flags)
    elif path == "camera":
        state = _trace_state(cw.Scene(_layout(W.c1_mesh(seed))), _camera_rays(case), flags | cw.TRACE_PRIM_ID)
    elif path == "frame":
        mesh = W.c1_mesh(seed)
        state = _trace_state(cw.Scene(_layout(mesh, case["kind"])), _frame_rays(case, mesh, g), flags)
    elif path == "bound":
        mesh = _mesh(case["mesh"], case["triangles"], seed)
        lay = _layout(mesh)
        state = _trace_state(None, _ao_rays(mesh, case["rays"], g), flags)
        state["arrays"] = [torch.from_numpy(a).cuda() for a in (lay.nodes, lay.woop, lay.prim_idx)]
        cw.set_log(False)
    elif path == "surfels":
        mesh = _mesh(case["mesh"], case["triangles"], seed)
        p, nrm = _surface(mesh, case["surfels"], g, in_order=True)
        diag = mesh.diagonal()
        pad = torch.zeros((len(p), 1), device="cuda")
        state = {"scene": cw.Scene(_layout(mesh)), "pos": torch.cat((p, pad), 1), "nrm": torch.cat((nrm, pad), 1),
                 "rad": torch.full((len(p),), 2e-4 * diag, device="cuda"), "tmax": 0.05 * diag, "seed": int(seed),
                 "spp": case["spp"], "flags": flags, "counts": torch.empty(len(p), dtype=torch.int32, device="cuda")}
    elif path == "batch":
        plan, rng = _plan(case, seed)
        scenes = _scenes(plan)
        counts = [int(math.exp(rng.uniform(math.log(1000), math.log(case["max_rays"])))) for _ in scenes]
        rays = torch.cat([_ao_rays(mesh, n, g) for (mesh, _), n in zip(scenes, counts)])
        hits = torch.empty((len(rays), 4), device="cuda")
        items, first = [], 0
        for (_, scene), n in zip(scenes, counts):
            items.append((scene, rays.data_ptr() + 32 * first, hits.data_ptr() + 16 * first, n))
            first += n
        stream = cw.Stream()
        batch = cw.Batch(items, flags)
        batch.capture(stream)
        state = {"batch": batch, "stream": stream, "rays": rays, "hits": hits}
    else:
        plan, rng = _plan(case, seed)
        scenes = _scenes(plan)
        pool = [_ao_rays(mesh, case["max_rays"], g) for mesh, _ in scenes]
        counts = np.exp(rng.uniform(math.log(1000), math.log(case["max_rays"]), case["requests"])).astype(np.int64)
        which = rng.integers(0, len(scenes), case["requests"])
        first = np.concatenate(([0], np.cumsum(counts)))
        state = {"server": cw.Server([s for _, s in scenes], cw.default_server_config(flags=flags)),
                 "scenes": scenes, "pool": pool, "hits": torch.empty((int(first[-1]), 4), device="cuda"),
                 "requests": [(int(k), pool[k].data_ptr(), int(n), int(f)) for k, n, f in zip(which, counts, first)]}
    state["path"] = path
    torch.cuda.synchronize()
    return state


def _hits(h):
    return {"t": h[:, 0], "triangle": h.view(torch.int32)[:, 1], "uv": h[:, 2:4]}


def run(s):
    path = s["path"]
    if path == "surfels":
        s["counts"].zero_()
        s["scene"].trace_surfels(s["pos"].data_ptr(), s["nrm"].data_ptr(), s["rad"].data_ptr(), len(s["rad"]),
                                 s["spp"], 0.0, s["tmax"], s["seed"], s["flags"],
                                 d_texel_hits=s["counts"].data_ptr())
        return s["counts"]
    if path == "batch":
        s["batch"].replay(s["stream"])
    elif path == "server":
        out = s["hits"].data_ptr()
        for scene, rays, n, first in s["requests"]:
            s["server"].submit_device(scene, rays, n, out + 16 * first)
        s["server"].drain()
    elif path == "bound":
        nodes, woop, prim = s["arrays"]
        cw.rtBindCWBVHData(nodes.data_ptr(), woop.data_ptr(), prim.data_ptr())
        cw.rtTraceCWBVH(s["rays"].data_ptr(), s["hits"].data_ptr(), len(s["rays"]))
    else:
        s["scene"].trace(s["rays"].data_ptr(), s["hits"].data_ptr(), len(s["rays"]), s["flags"])
    return _hits(s["hits"])


def work(case):
    """Rays read and hits written once, the scene read once; the slab and
    triangle tests of the visits a ray cannot avoid."""
    path = case["path"]
    out = 16
    if path == "trace" or path == "bound":
        rays, tris, mesh = case["rays"], case["triangles"], case["mesh"]
    elif path == "camera":
        rays, tris, mesh = case["width"] * case["height"], 980002, "spheres"
    elif path == "frame":
        rays, tris, mesh = case["width"] * case["height"] * case["spp"], 980002, "spheres"
    elif path == "surfels":
        rays, tris, mesh = case["surfels"] * case["spp"], case["triangles"], case["mesh"]
    else:
        # log-uniform sizes between 1000 and the largest
        def mean(hi):
            return (hi - 1000) / math.log(hi / 1000)

        tris, mesh = int(case["scenes"] * mean(case["max_triangles"])), "spheres"
        rays = int(mean(case["max_rays"]) * (case["scenes"] if path == "batch" else case["requests"]))
    nodes, tests = VISITS[mesh]
    # a slab test is 6 fused multiply-adds, a triangle test about 50 operations
    slabs = nodes * (2.8 * 2 if case.get("kind") == "bvh2" else 8)
    moved = 40 * case["surfels"] if path == "surfels" else (32 + out) * rays
    return {"bytes": moved + min(tris, rays * 8) * 60, "flops": rays * (slabs * 12 + tests * 50)}


# --------------------------------------------------------- 64-bit reference


def exact(case, seed):
    """Closest hits of a small single trace by testing every triangle in
    64 bits; nothing for larger cases, any hit (whose triangle is free) and
    the integer outputs."""
    if case["path"] not in ("trace", "bound") or case.get("mode", "closest") != "closest":
        return None
    if case["rays"] * case["triangles"] > 1 << 31 or case["mesh"] == "soup":
        return None
    mesh = _mesh(case["mesh"], case["triangles"], seed)
    rays = _ao_rays(mesh, case["rays"], _generator(seed)).double()
    a, b, c = (x.double() for x in _corners(mesh))
    # barycentric weights of the corners a and b (the third is c), as the hits report them
    e1, e2 = a - c, b - c
    step = max(1, (1 << 26) // len(a))
    t_all, uv_all = [], []
    for k in range(0, len(rays), step):
        o, tmin, d, tmax = rays[k:k + step, None, 0:3], rays[k:k + step, 3:4], rays[k:k + step, None, 4:7], rays[k:k + step, 7:8]
        h = torch.linalg.cross(d.expand(-1, len(a), -1), e2.expand(len(d), -1, -1))
        det = (e1 * h).sum(2)
        s = o - c
        u = (s * h).sum(2) / det
        del h
        q = torch.linalg.cross(s, e1.expand(len(d), -1, -1))
        del s
        v = (d * q).sum(2) / det
        t = (e2 * q).sum(2) / det
        del q
        ok = (det != 0) & (u >= 0) & (v >= 0) & (u + v <= 1) & (t > tmin) & (t < tmax)
        t = torch.where(ok, t, math.inf)
        best, at = t.min(dim=1, keepdim=True)
        miss = torch.isinf(best)
        t_all.append(torch.where(miss, tmax, best)[:, 0])
        uv = torch.cat((u.gather(1, at), v.gather(1, at)), 1)
        uv_all.append(torch.where(miss, 0.0, uv))
    return {"t": torch.cat(t_all), "triangle": None, "uv": torch.cat(uv_all)}
