"""The last rays of a wave, traced with teams of 4 or 8 lanes per ray: hits are
bit-identical to the scalar oracle at every size where the division of lanes
changes (rays per wave 8, 16 and 64; 16 and 8 rays left; ragged last waves)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 8 rays per wave up to 8 x 16 x 256 = 32,768 rays, 16 up to 65,536, then 64
SIZES = [1, 7, 8, 9, 15, 16, 17, 63, 64, 65, 129, 4095, 32767, 32768, 32769, 65535, 65536, 65537, 70001]


def bits(h):
    return np.ascontiguousarray(h, np.float32).view(np.uint32)


@pytest.fixture(scope="module", params=["spheres", "soup"])
def scene(request, cw, orc):
    """A lattice of spheres under AO rays, and a soup (up to 3 triangles per
    leaf, many per node) under unbounded rays, with the oracle's hits."""
    if request.param == "spheres":
        mesh = cw.Mesh.icosphere_grid(4, 4, 4, 6, 4.0, 0.5, 1.5, 1.0, seed=11)
        rays = cw.rays_ao_surface(mesh, (SIZES[-1] + 7) // 8, 8, 1e-4 * mesh.diagonal(), 0.0, 0.1 * mesh.diagonal(), seed=12)
    else:
        mesh = cw.Mesh.cluster_soup(40000, 64, 0.02, 0.1, -4.0, 0.5, seed=13)
        rays = cw.rays_sphere_from_surface(mesh, SIZES[-1], 1e-4 * mesh.diagonal(), seed=14)
    rays = rays[:SIZES[-1]]
    _, lay = cw.build_layouts(mesh, bvh2=False)
    refs = {a: bits(orc.trace_cwbvh(lay.nodes, lay.node_stride, lay.woop, rays, any_hit=a)) for a in (False, True)}
    return cw.Scene(lay), rays, refs


@pytest.mark.parametrize("any_hit", [False, True])
def test_every_division_of_lanes(cw, scene, any_hit):
    sc, rays, refs = scene
    for n in SIZES:
        print(f"[gpu-test] teams n={n} any={any_hit}", flush=True)
        got = bits(sc.trace_numpy(rays[:n], cw.TRACE_ANY if any_hit else cw.TRACE_CLOSEST))
        assert np.array_equal(got, refs[any_hit][:n]), n


@pytest.mark.parametrize("cfg", [dict(persistent=1), dict(persistent=1, grid_blocks=5, fetch_chunk=7),
                                 dict(persistent=1, occupancy=7), dict(persistent=1, prefetch=1),
                                 dict(persistent=0, block_size=256), dict(persistent=0, block_size=64, prefetch=1)])
@pytest.mark.parametrize("any_hit", [False, True])
def test_ends_of_persistent_waves(cw, scene, cfg, any_hit):
    sc, rays, refs = scene
    for n in (5, 257, 20001):
        print(f"[gpu-test] teams {cfg} n={n} any={any_hit}", flush=True)
        got = bits(sc.trace_numpy(rays[:n], cw.TRACE_ANY if any_hit else cw.TRACE_CLOSEST, sc.default_config(**cfg)))
        assert np.array_equal(got, refs[any_hit][:n]), n


@pytest.mark.parametrize("any_hit", [False, True])
def test_jobs_of_a_batch_share_waves(cw, scene, any_hit):
    """Teams of one wave hold rays of different scenes and jobs."""
    sc, rays, refs = scene
    other = cw.Mesh.heightfield(40, 30, 4, 0.2, seed=15)
    sc2 = cw.Scene(cw.build_layouts(other, bvh2=False)[1])
    counts = [3, 20, 1, 64, 300]
    bufs, items = [], []
    first = 0
    for n in counts:
        for s in (sc, sc2):
            dr, dh = cw.DeviceBuffer.from_numpy(rays[first:first + n]), cw.DeviceBuffer(16 * n)
            bufs.append((dr, dh, first, n, s))
            items.append((s, dr.ptr, dh.ptr, n))
        first += n
    batch = cw.Batch(items, cw.TRACE_ANY if any_hit else cw.TRACE_CLOSEST)
    print(f"[gpu-test] teams batch any={any_hit}", flush=True)
    batch.launch()
    cw.synchronize()
    for dr, dh, f, n, s in bufs:
        if s is sc:
            assert np.array_equal(bits(dh.download((n, 4))), refs[any_hit][f:f + n]), n


@pytest.mark.parametrize("any_hit", [False, True])
def test_four_rays_per_wave(cw, scene, any_hit):
    """4 rays per wave up to 4 x 2 x 256 = 2,048 rays, then 8."""
    sc, rays, refs = scene
    for n in (2, 3, 4, 5, 2044, 2047, 2048, 2049, 2056):
        print(f"[gpu-test] four per wave n={n} any={any_hit}", flush=True)
        got = bits(sc.trace_numpy(rays[:n], cw.TRACE_ANY if any_hit else cw.TRACE_CLOSEST))
        assert np.array_equal(got, refs[any_hit][:n]), n
