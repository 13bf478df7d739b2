"""The bound trace and the null stream's overflow flag: an overflow that an
earlier launch left there is reported and not taken for the bound trace's own,
and a thread that reads the flag during a bound trace neither changes its hits
nor is told of an overflow that a valid tree does not have."""
import threading

import numpy as np
import pytest

from test_gpu_bound import bits, deep_mesh

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def deep(cw, orc):
    """A chain-like tree of more than 13 stack entries, and rays down the chain."""
    rng = np.random.default_rng(51)
    n = 20000
    to = (0.8 ** rng.uniform(0, 300, n))[:, None] * np.array([1.0, 0.03, 0.03])
    o = np.array([3.0, 0.0, 0.0]) + rng.uniform(-0.02, 0.02, (n, 3))
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3], rays[:, 4:7], rays[:, 7] = o, to - o, np.inf
    _, lay = cw.build_layouts(deep_mesh(cw), bvh2=False)
    assert 13 < lay.stats()["stack_need"] <= 64
    bufs = [cw.DeviceBuffer.from_numpy(a) for a in (lay.nodes, lay.woop, lay.prim_idx)]
    return bufs, rays, bits(orc.trace_cwbvh(lay.nodes, lay.node_stride, lay.woop, rays)), lay


def test_a_pending_overflow_is_reported(cw, deep):
    bufs, rays, ref, lay = deep
    cw.set_log(False)
    d_rays, d_hits = cw.DeviceBuffer.from_numpy(rays), cw.DeviceBuffer(16 * len(rays))
    cw.rtBindCWBVHData(*(b.ptr for b in bufs))
    cw.stack_overflowed()
    # arrays wrapped with a smaller need than the tree's: the launch overflows and says so in the flag
    small = cw.Scene.wrap(lay.kind, lay.node_stride, bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, 4, keep=bufs)
    small.trace(d_rays.ptr, d_hits.ptr, len(rays), cw.TRACE_CLOSEST, small.default_config(lds_depth=4))
    print("[gpu-test] pending overflow", flush=True)
    with pytest.raises(cw.CwbvhError, match="stack overflow"):
        cw.rtTraceCWBVH(d_rays.ptr, d_hits.ptr, len(rays))
    # reported once; the bound trace's own hits are complete
    assert np.array_equal(bits(d_hits.download((len(rays), 4))), ref)
    cw.rtTraceCWBVH(d_rays.ptr, d_hits.ptr, len(rays))
    cw.set_log(True)


def test_a_thread_that_reads_the_flag(cw, deep):
    bufs, rays, ref, _ = deep
    cw.set_log(False)
    d_rays, d_hits = cw.DeviceBuffer.from_numpy(rays), cw.DeviceBuffer(16 * len(rays))
    cw.stack_overflowed()
    stop, seen = threading.Event(), []

    def poll():
        while not stop.is_set():
            seen.append(cw.stack_overflowed())

    t = threading.Thread(target=poll)
    t.start()
    try:
        for _ in range(60):
            cw.rtBindCWBVHData(*(b.ptr for b in bufs))
            d_hits.zero()
            cw.rtTraceCWBVH(d_rays.ptr, d_hits.ptr, len(rays))
            assert np.array_equal(bits(d_hits.download((len(rays), 4))), ref)
    finally:
        stop.set()
        t.join()
        cw.set_log(True)
    print(f"[gpu-test] flag read {len(seen)} times during 60 bound traces", flush=True)
    assert seen and not any(seen)
