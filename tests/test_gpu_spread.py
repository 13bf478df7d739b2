"""Scenes with 128 B nodes are traversed on nodes whose 16-byte slots are
exchanged by the node's index: hits are bit-identical to the oracle for trees
of one node and more, whatever the node count leaves of the last eight."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bits(h):
    return np.ascontiguousarray(h, np.float32).view(np.uint32)


@pytest.mark.parametrize("tris", [1, 2, 9, 60, 61, 64, 333, 20000])
@pytest.mark.parametrize("any_hit", [False, True])
def test_spread_nodes(cw, orc, tris, any_hit):
    mesh = cw.Mesh.cluster_soup(tris, 8, 0.05, 0.2, -2.5, 0.5, seed=tris)
    diag = mesh.diagonal()
    rays = cw.rays_sphere_from_surface(mesh, 3001, 1e-4 * diag, seed=tris + 1)
    _, lay = cw.build_layouts(mesh, bvh2=False)
    ref = bits(orc.trace_cwbvh(lay.nodes, lay.node_stride, lay.woop, rays, any_hit=any_hit))
    flags = cw.TRACE_ANY if any_hit else cw.TRACE_CLOSEST
    for sc in (cw.Scene(lay, stride_mode=cw.SCENE_STRIDE_128), cw.Scene(lay.restride(8))):
        assert sc.node_stride == 8
        for cfg in ({}, dict(persistent=1), dict(persistent=1, prefetch=1), dict(persistent=0, prefetch=1),
                    dict(persistent=1, occupancy=7), dict(loop_mode=0), dict(loop_mode=2, prefetch=1),
                    dict(persistent=1, prefetch=1, refill_idle=0, refill_budget=1, fetch_chunk=3)):
            print(f"[gpu-test] spread tris={tris} any={any_hit} {cfg}", flush=True)
            got = bits(sc.trace_numpy(rays, flags, sc.default_config(**cfg)))
            if cfg.get("loop_mode") == 2 and any_hit:
                # speculation reorders triangle tests: occlusion only
                assert np.array_equal(got[:, 1] == 0xFFFFFFFF, ref[:, 1] == 0xFFFFFFFF), cfg
            else:
                assert np.array_equal(got, ref), cfg
