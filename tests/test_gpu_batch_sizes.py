"""Batches at the sizes where the plan changes: chunks of 8, 16 and 64 rays,
more chunks than waves, one job to more jobs than lanes (the chunk search's
segments), against the oracle bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bits(h):
    return np.ascontiguousarray(h, np.float32).view(np.uint32)


@pytest.fixture(scope="module")
def data(cw, orc):
    mesh = cw.Mesh.icosphere_grid(3, 3, 3, 5, 4.0, 0.5, 1.5, 1.0, seed=21)
    diag = mesh.diagonal()
    rays = cw.rays_ao_surface(mesh, 45000, 8, 1e-4 * diag, 0.0, 0.15 * diag, seed=22)
    _, lay = cw.build_layouts(mesh, bvh2=False)
    refs = {a: bits(orc.trace_cwbvh(lay.nodes, lay.node_stride, lay.woop, rays, any_hit=a)) for a in (False, True)}
    return cw.Scene(lay), rays, refs, cw.DeviceBuffer.from_numpy(rays)


# total rays: 8 per wave to 32,768, 16 to 65,536, then 64; jobs: 64 fit the lanes
@pytest.mark.parametrize("jobs", [1, 2, 63, 64, 65, 127, 128, 129, 700])
@pytest.mark.parametrize("total", [701, 32768, 32769, 65537, 360000])
@pytest.mark.parametrize("any_hit", [False, True])
def test_every_plan(cw, data, jobs, total, any_hit):
    sc, rays, refs, d_rays = data
    rng = np.random.default_rng([jobs, total])
    cuts = np.sort(rng.choice(np.arange(1, total), jobs - 1, replace=False))
    edges = np.concatenate(([0], cuts, [total]))
    d_hits = cw.DeviceBuffer(16 * total)
    d_hits.zero()
    items = [(sc, d_rays.ptr + 32 * int(a), d_hits.ptr + 16 * int(a), int(b - a)) for a, b in zip(edges, edges[1:])]
    batch = cw.Batch(items, cw.TRACE_ANY if any_hit else cw.TRACE_CLOSEST)
    print(f"[gpu-test] batch jobs={jobs} total={total} any={any_hit}", flush=True)
    for _ in range(2):   # the counters are reset for the next launch
        batch.launch()
    cw.synchronize()
    assert np.array_equal(bits(d_hits.download((total, 4))), refs[any_hit][:total])


def test_server_refuses_more_scenes_than_its_table(cw, data):
    sc = data[0]
    with pytest.raises(cw.CwbvhError, match="too many scenes"):
        cw.Server([sc] * 4097)
