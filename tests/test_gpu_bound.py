"""Trees whose stack need is unknown (bound or wrapped arrays): the kernels with
a two-level stack, their teams of lanes, and the bound trace that first assumes
a shallow tree, on a tree far deeper than it assumes and on an ordinary one.
Rays along the deep tree's chain of triangles graze many edges, so their hits
also show whether ties are settled as in the oracle, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 8, 9, 17, 64, 65, 1000, 32769, 66000, 900000]


def bits(h):
    return np.ascontiguousarray(h, np.float32).view(np.uint32)


def deep_mesh(cw):
    """Triangles shrinking towards the origin: every split separates a few of
    the largest, so the tree is a chain."""
    s = 0.8 ** np.arange(400)
    v = np.zeros((400, 3, 3), np.float32)
    v[:, 0, 0], v[:, 1, 0], v[:, 1, 1], v[:, 2, 0], v[:, 2, 2] = s, 1.05 * s, 0.1 * s, 1.05 * s, 0.1 * s
    return cw.Mesh.from_arrays(v.reshape(-1, 3), np.arange(1200, dtype=np.int32).reshape(-1, 3))


@pytest.fixture(scope="module", params=["deep", "spheres"])
def bound(request, cw, orc):
    rng = np.random.default_rng(31)
    n = SIZES[-1]
    if request.param == "deep":
        mesh = deep_mesh(cw)
        # towards points of the chain, from beyond its large end and from the side
        to = (0.8 ** rng.uniform(0, 300, n))[:, None] * np.array([1.0, 0.03, 0.03])
        o = np.array([3.0, 0.0, 0.0]) + rng.uniform(-0.02, 0.02, (n, 3)) * np.array([1, 1, 1])
        rays = np.zeros((n, 8), np.float32)
        rays[:, 0:3], rays[:, 4:7], rays[:, 7] = o, to - o, np.inf
    else:
        mesh = cw.Mesh.icosphere_grid(3, 3, 3, 5, 4.0, 0.5, 1.5, 1.0, seed=32)
        rays = cw.rays_ao_surface(mesh, n // 8 + 1, 8, 1e-4 * mesh.diagonal(), 0.0, 0.1 * mesh.diagonal(), seed=33)[:n]
    _, lay = cw.build_layouts(mesh, bvh2=False)
    bufs = [cw.DeviceBuffer.from_numpy(a) for a in (lay.nodes, lay.woop, lay.prim_idx)]
    refs = {a: bits(orc.trace_cwbvh(lay.nodes, lay.node_stride, lay.woop, rays, any_hit=a)) for a in (False, True)}
    return request.param, lay, bufs, rays, refs


def wrap(cw, bound, need):
    _, lay, bufs, _, _ = bound
    return cw.Scene.wrap(lay.kind, lay.node_stride, bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, need, keep=bufs)


def test_the_deep_tree_is_deep(cw, bound):
    name, lay, _, rays, _ = bound
    sc = wrap(cw, bound, 13)   # a need that the tree exceeds
    cw.stack_overflowed()
    print(f"[gpu-test] bound depth {name}", flush=True)
    sc.trace_numpy(rays[:1000], cw.TRACE_CLOSEST, sc.default_config(lds_depth=13))
    assert cw.stack_overflowed() == (name == "deep")


@pytest.mark.parametrize("any_hit", [False, True])
def test_unknown_need(cw, bound, any_hit):
    name, _, _, rays, refs = bound
    sc = wrap(cw, bound, 0)
    for n in SIZES:
        for cfg in ({}, dict(lds_depth=1), dict(lds_depth=3, persistent=1), dict(lds_depth=2, prefetch=1)):
            print(f"[gpu-test] unknown need {name} n={n} any={any_hit} {cfg}", flush=True)
            got = bits(sc.trace_numpy(rays[:n], cw.TRACE_ANY if any_hit else cw.TRACE_CLOSEST, sc.default_config(**cfg)))
            assert np.array_equal(got, refs[any_hit][:n]), (n, cfg)
    assert not cw.stack_overflowed()


@pytest.mark.parametrize("any_hit", [False, True])
def test_built_scene(cw, bound, any_hit):
    """The same scene with its need known: stack in LDS only, with and without
    work fetching and node prefetch."""
    name, lay, _, rays, refs = bound
    sc = cw.Scene(lay)
    for n in SIZES:
        for cfg in ({}, dict(persistent=0), dict(prefetch=1), dict(occupancy=7)):
            print(f"[gpu-test] built scene {name} n={n} any={any_hit} {cfg}", flush=True)
            got = bits(sc.trace_numpy(rays[:n], cw.TRACE_ANY if any_hit else cw.TRACE_CLOSEST, sc.default_config(**cfg)))
            assert np.array_equal(got, refs[any_hit][:n]), (n, cfg)


def test_bound_trace(cw, bound):
    name, _, bufs, rays, refs = bound
    cw.set_log(False)
    d_rays = cw.DeviceBuffer.from_numpy(rays)
    for n in SIZES:
        d_hits = cw.DeviceBuffer(16 * n)
        cw.rtBindCWBVHData(*(b.ptr for b in bufs))
        for _ in range(2):   # the second trace knows the tree
            print(f"[gpu-test] bound trace {name} n={n}", flush=True)
            d_hits.zero()
            cw.rtTraceCWBVH(d_rays.ptr, d_hits.ptr, n)
            assert np.array_equal(bits(d_hits.download((n, 4))), refs[False][:n]), n
    cw.set_log(True)
