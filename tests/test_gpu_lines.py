"""The default launches of each kind on both sides of every ray count where the
dispatch changes the kernel, the grid or the block, bit for bit against the
oracle.  The rays of a small set are repeated to fill the launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PERSISTENT, PERSISTENT_ANY = 3 << 18, 5 << 18
SORTED = 1 << 20
SEVEN_WAVES = 3 << 21
BVH2_L2_BLOCKS, BVH2_BLOCKS = 1 << 20, 3 << 23


def bits(h):
    return np.ascontiguousarray(h, np.float32).view(np.uint32)


def around(*lines):
    return [n + k for n in lines for k in (-1, 0, 1)]


class Set:
    """A scene of each kind, base rays with their hits, and the base rays repeated to `n` on the device."""

    def __init__(self, cw, orc, n):
        mesh = cw.Mesh.icosphere_grid(5, 5, 4, 6, 4.0, 0.5, 1.5, 1.0, seed=71)
        rays = cw.rays_ao_surface(mesh, 12000, 8, 1e-4 * mesh.diagonal(), 0.0, 0.1 * mesh.diagonal(), seed=72)[:95003]
        self.bvh2, self.cwbvh = cw.build_layouts(mesh)
        self.refs = {("cwbvh", a): bits(orc.trace_cwbvh(self.cwbvh.nodes, self.cwbvh.node_stride, self.cwbvh.woop, rays, any_hit=a)) for a in (False, True)}
        self.refs.update({("bvh2", a): bits(orc.trace_bvh2(self.bvh2.nodes, self.bvh2.woop, rays, any_hit=a)) for a in (False, True)})
        self.cw, self.rays, self.n = cw, rays, 0
        self.grow(n)

    def grow(self, n):
        if n > self.n:
            reps = -(-n // len(self.rays))
            self.d_rays = self.cw.DeviceBuffer.from_numpy(np.tile(self.rays, (reps, 1)))
            self.d_hits = self.cw.DeviceBuffer(16 * reps * len(self.rays))
            self.n = reps * len(self.rays)

    def check(self, kind, any_hit, n, launch, what, same=lambda h: h):
        print(f"[gpu-test] lines {kind} {what} n={n} any={any_hit}", flush=True)
        launch(n, self.cw.TRACE_ANY if any_hit else self.cw.TRACE_CLOSEST)
        self.cw.synchronize()
        got, ref = same(bits(self.d_hits.download((n, 4)))), same(self.refs[kind, any_hit])
        for k in range(0, n, len(ref)):
            assert np.array_equal(got[k:k + len(ref)], ref[:n - k]), (what, n, k)


@pytest.fixture(scope="module")
def rays(cw, orc):
    return Set(cw, orc, SEVEN_WAVES + 1)


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("cfg", [{}, dict(loop_mode=0), dict(loop_mode=2)])
def test_cwbvh_in_the_cache(cw, rays, cfg, any_hit):
    sc = cw.Scene(rays.cwbvh)
    # which accepted triangle ends a speculative any-hit ray is open: there, hit or miss
    same = (lambda h: h[:, 1] != 0xFFFFFFFF) if any_hit and cfg.get("loop_mode") == 2 else (lambda h: h)
    for n in around(PERSISTENT, PERSISTENT_ANY, SEVEN_WAVES):
        rays.check("cwbvh", any_hit, n, lambda n, fl: sc.trace(rays.d_rays.ptr, rays.d_hits.ptr, n, fl, sc.default_config(**cfg)), cfg, same)


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("cfg", [{}, dict(ray_order=0), dict(loop_mode=0, prefetch=0, ray_order=0)])
def test_cwbvh_that_streams(cw, rays, cfg, any_hit):
    """Arrays in an allocation larger than the Infinity Cache count as a scene of that size."""
    lay = rays.cwbvh
    nodes = np.zeros((300 << 20) // 16 * 4, np.float32)
    flat = np.ascontiguousarray(lay.nodes, np.float32).reshape(-1)
    nodes[:len(flat)] = flat
    bufs = [cw.DeviceBuffer.from_numpy(a) for a in (nodes, lay.woop, lay.prim_idx)]
    sc = cw.Scene.wrap(lay.kind, lay.node_stride, bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, lay.stats()["stack_need"], keep=bufs)
    assert sc.device_bytes() > 256 << 20 and sc.default_config().prefetch == 1
    for n in around(PERSISTENT, SORTED, PERSISTENT_ANY):
        rays.check("cwbvh", any_hit, n, lambda n, fl: sc.trace(rays.d_rays.ptr, rays.d_hits.ptr, n, fl, sc.default_config(**cfg)), cfg)


def test_bound_arrays(cw, rays):
    lay = rays.cwbvh
    bufs = [cw.DeviceBuffer.from_numpy(a) for a in (lay.nodes, lay.woop, lay.prim_idx)]
    cw.set_log(False)
    cw.rtBindCWBVHData(*(b.ptr for b in bufs))
    for n in around(PERSISTENT, SEVEN_WAVES):
        rays.check("cwbvh", False, n, lambda n, fl: cw.rtTraceCWBVH(rays.d_rays.ptr, rays.d_hits.ptr, n), "bound")
    cw.set_log(True)


@pytest.mark.parametrize("any_hit", [False, True])
def test_surfels(cw, orc, rays, any_hit):
    """2^21 rays (persistent grid) and 2^22 (7 waves), 16 per surfel: counts per surfel do not depend on the launch."""
    spp, most = 16, (1 << 18) + 1
    rng = np.random.default_rng(73)
    pos, nrm = np.zeros((most, 4), np.float32), np.zeros((most, 4), np.float32)
    at = rng.integers(0, len(rays.rays), most)
    pos[:, :3], nrm[:, :3] = rays.rays[at, 0:3], rays.rays[at, 4:7]
    nrm[:, :3] /= np.linalg.norm(nrm[:, :3], axis=1, keepdims=True)
    rad = np.full(most, 1e-3, np.float32)
    gen = cw.rays_ao_from_samples(pos, nrm, rad, spp, 0.0, np.float32(2.0), seed=74)
    hit = orc.trace_cwbvh(rays.cwbvh.nodes, rays.cwbvh.node_stride, rays.cwbvh.woop, gen, any_hit=any_hit)
    ref = (cw.hit_ids(hit) >= 0).reshape(most, spp).sum(1).astype(np.uint32)
    sc, bufs, counts = cw.Scene(rays.cwbvh), [cw.DeviceBuffer.from_numpy(a) for a in (pos, nrm, rad)], cw.DeviceBuffer(4 * most)
    for m in around(1 << 17, 1 << 18):
        print(f"[gpu-test] lines surfels {m * spp} rays any={any_hit}", flush=True)
        counts.zero()
        sc.trace_surfels(bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, m, spp, 0.0, 2.0, 74, cw.TRACE_ANY if any_hit else cw.TRACE_CLOSEST, d_texel_hits=counts.ptr)
        cw.synchronize()
        assert np.array_equal(counts.download((most,), np.uint32)[:m], ref[:m]), m


@pytest.mark.parametrize("any_hit", [False, True])
def test_bvh2(cw, rays, any_hit):
    sc = cw.Scene(rays.bvh2)
    assert sc.device_bytes() > 4 << 20
    rays.grow(BVH2_BLOCKS + 1)
    for n in around(BVH2_L2_BLOCKS, BVH2_BLOCKS):
        rays.check("bvh2", any_hit, n, lambda n, fl: sc.trace(rays.d_rays.ptr, rays.d_hits.ptr, n, fl), "default")


@pytest.mark.parametrize("any_hit", [False, True])
def test_unknown_need(cw, rays, any_hit):
    """Arrays of unknown stack need: any hit runs 7 waves from 2^22 rays up, closest hit from 3 x 2^21."""
    lay = rays.cwbvh
    bufs = [cw.DeviceBuffer.from_numpy(a) for a in (lay.nodes, lay.woop, lay.prim_idx)]
    sc = cw.Scene.wrap(lay.kind, lay.node_stride, bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, 0, keep=bufs)
    for n in around(1 << 22, SEVEN_WAVES):
        rays.check("cwbvh", any_hit, n, lambda n, fl: sc.trace(rays.d_rays.ptr, rays.d_hits.ptr, n, fl), "unknown need")
    assert not cw.stack_overflowed()
