"""Small requests beside a large one: while a launch of many rays is in flight
and slots are free, a small host or device request gets a launch of its own
instead of waiting for the large one to end."""
import numpy as np
import pytest

from test_gpu_serving import bits, oracle_hits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def large(cw):
    """A scene, 250,000 rays in pinned memory with their hits, and the same rays 48 times over on the device."""
    from cwbvh_amd import workloads as W

    mesh = W.icospheres_of(60000, seed=310)
    _, lay = cw.build_layouts(mesh, bvh2=False)
    rays = cw.rays_ao_surface(mesh, 31250, 8, 1e-4 * mesh.diagonal(), 0.0, 0.1 * mesh.diagonal(), seed=311)
    pool = cw.PinnedArray(rays.shape, np.float32)
    pool.array[:] = rays
    return cw.Scene(lay), pool, bits(oracle_hits(lay, rays)), cw.DeviceBuffer.from_numpy(np.tile(rays, (48, 1)))


@pytest.mark.parametrize("kind", ["host", "device"])
def test_small_requests_do_not_wait_for_a_large_one(cw, large, kind):
    scene, pool, ref, d_rays = large
    n, small = 48 * len(ref), 3000
    d_hits = cw.DeviceBuffer(16 * n)
    srv = cw.Server([scene], cw.default_server_config(memory_budget=64 << 20))
    print(f"[gpu-test] {n} rays in flight, then a {kind} request of {small}", flush=True)
    out = cw.PinnedArray((small, 4), np.float32) if kind == "host" else cw.DeviceBuffer(16 * small)
    first = srv.submit_device(0, d_rays.ptr, n, d_hits.ptr)
    while srv.stats()["batches"] == 0:   # launched: the next request cannot share its launch
        pass
    if kind == "host":
        second = srv.submit(0, pool.ptr, small, out.ptr)
    else:
        second = srv.submit_device(0, d_rays.ptr, small, out.ptr)
    srv.wait(second, 60.0)
    srv.wait(first, 60.0)
    st = srv.stats()
    srv.close()
    got = out.array if kind == "host" else out.download((small, 4))
    assert np.array_equal(bits(got), ref[:small])
    assert np.array_equal(bits(d_hits.download((n, 4))), np.tile(ref, (48, 1)))
    assert st["max_inflight_seen"] > 1, st
