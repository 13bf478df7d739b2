"""BVH2 launches with one ray per lane: 1, 2, 4, 8, 16 or 64 rays per wave by the
launch's size (at most 16 waves per compute unit below 64).  Hits are
bit-identical to the scalar oracle around every change of the share."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 16 waves x 256 units = 4096 waves: shares change at 4096 x 1, 2, 4, 8, 16 rays
SIZES = [1, 2, 63, 64, 65, 4095, 4096, 4097, 8192, 8193, 16384, 16385, 32768, 32769, 65536, 65537, 70003]


def bits(h):
    return np.ascontiguousarray(h, np.float32).view(np.uint32)


@pytest.fixture(scope="module", params=["spheres", "soup"])
def scene(request, cw, orc):
    if request.param == "spheres":
        mesh = cw.Mesh.icosphere_grid(4, 4, 4, 6, 4.0, 0.5, 1.5, 1.0, seed=41)
        rays = cw.rays_ao_surface(mesh, (SIZES[-1] + 7) // 8, 8, 1e-4 * mesh.diagonal(), 0.0, 0.1 * mesh.diagonal(), seed=42)
    else:
        mesh = cw.Mesh.cluster_soup(40000, 64, 0.02, 0.1, -4.0, 0.5, seed=43)
        rays = cw.rays_sphere_from_surface(mesh, SIZES[-1], 1e-4 * mesh.diagonal(), seed=44)
    rays = rays[:SIZES[-1]]
    lay, _ = cw.build_layouts(mesh, cwbvh=False)
    refs = {a: bits(orc.trace_bvh2(lay.nodes, lay.woop, rays, any_hit=a)) for a in (False, True)}
    return cw.Scene(lay), rays, refs


@pytest.mark.parametrize("cfg", [{}, dict(block_size=64, lds_depth=1), dict(block_size=128, lds_depth=3)])
@pytest.mark.parametrize("any_hit", [False, True])
def test_every_share(cw, scene, any_hit, cfg):
    sc, rays, refs = scene
    for n in SIZES:
        print(f"[gpu-test] bvh2 share n={n} any={any_hit} {cfg}", flush=True)
        got = bits(sc.trace_numpy(rays[:n], cw.TRACE_ANY if any_hit else cw.TRACE_CLOSEST, sc.default_config(**cfg)))
        assert np.array_equal(got, refs[any_hit][:n]), n


@pytest.mark.parametrize("any_hit", [False, True])
def test_blocks_of_a_scene_in_l2(cw, orc, any_hit):
    """A scene of up to 4 MB: blocks of block_size threads from 2^20 rays up."""
    mesh = cw.Mesh.heightfield(60, 40, 5, 0.1, seed=45)
    lay, _ = cw.build_layouts(mesh, cwbvh=False)
    sc = cw.Scene(lay)
    assert sc.device_bytes() <= 4 << 20
    n = (1 << 20) + 65
    rays = cw.rays_ao_surface(mesh, (n + 7) // 8, 8, 1e-4 * mesh.diagonal(), 0.0, 0.1 * mesh.diagonal(), seed=46)[:n]
    ref = bits(orc.trace_bvh2(lay.nodes, lay.woop, rays, any_hit=any_hit))
    for m, cfg in ((n, {}), ((1 << 20) - 1, {}), (1 << 20, dict(block_size=128)), (n, dict(block_size=64, lds_depth=2))):
        print(f"[gpu-test] bvh2 in L2 n={m} any={any_hit} {cfg}", flush=True)
        got = bits(sc.trace_numpy(rays[:m], cw.TRACE_ANY if any_hit else cw.TRACE_CLOSEST, sc.default_config(**cfg)))
        assert np.array_equal(got, ref[:m]), (m, cfg)
