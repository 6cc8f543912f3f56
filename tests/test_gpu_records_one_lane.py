"""Records from the one-lane-per-ray kernel at sizes where eight lanes are the default:
its record rings and slab rows, its stacks of four groups per list (treelet order) and
of 4, 8 and 16, their spills, and the finishing launches behind it.  Exact by contract,
so equal to the oracle's bit for bit."""
import numpy as np
import pytest

from conftest import assert_hits_equal, assert_records_equal
from golden import tiny_scene
from test_gpu_nodes import _gaps, _internal_nodes, _nan_origins, _scales
from test_gpu_records import _rays, _two_depth_rays

pytestmark = pytest.mark.gpu

STACKS = (4, 8, 16)


def _check(gpu, oracle, arena, tlas, rays, mode, budget, options):
    part = oracle.Partition(arena, tlas, budget)
    h_ref, o_ref, r_ref = oracle.trace(arena, tlas, rays, mode=mode, partition=part)
    gpu.set_scene(arena, tlas)
    gpu.build_treelets(budget)
    for kw in options:
        h, o, r = gpu.trace(rays, mode=mode, records=True, lanes_per_ray=1, **kw)
        assert_hits_equal(h, h_ref, f"{kw}")
        assert_records_equal(o, r, o_ref, r_ref, f"{kw}")
    return o_ref


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n,short,slab", [(1, 0, 0), (63, 0, 7), (257, 0.5, 33), (8192, 0.5, 40), (8193, 0.5, 0),
                                          (12000, 1.0, 8), (20000, 0.2, 1024)])
def test_rows_and_batch_edges(gpu, rtx, oracle, instanced, mode, n, short, slab):
    scene, rays = instanced
    _check(gpu, oracle, scene.arena, scene.tlas_offset, _rays(rtx, rays, n, short, n + 2), mode, 1024,
           [dict(record_slab=slab, lds_stack=k) for k in STACKS])


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("shared", [0, 1])
def test_deep_stacks_spill(gpu, rtx, oracle, mode, shared):
    """600 overlapping spheres: a ray through them has thousands of records and, with a TLAS
    and a BLAS of four levels and more each, more groups waiting than a list holds in LDS."""
    d = rtx.workload_desc(rtx.WORKLOAD_INSTANCED_SPHERES, n_instances=600, slices=32, stacks=16, shared_blas=shared,
                          width=16, height=16, seed=12, box_size=0.5)
    scene = rtx.workload_scene(d)
    rays = rtx.primary_rays(d)
    for flags in (0, rtx.RAY_FLAG_OPAQUE, rtx.RAY_FLAG_OPAQUE | rtx.RAY_FLAG_TERMINATE_ON_FIRST_HIT):
        rays["flags"] = flags
        o = _check(gpu, oracle, scene.arena, scene.tlas_offset, rays, mode, 1024,
                   [dict(lds_stack=k) for k in STACKS] + [dict(refill=1, waves_per_cu=4), dict(refill=64, record_slab=1024)])
        assert flags or np.diff(o).min() > 2000


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("budget", [256, 8192, 1 << 17])
def test_treelet_sizes_and_claims(gpu, rtx, oracle, c1, mode, budget):
    scene, rays = c1
    order = np.random.default_rng(budget).permutation(len(rays)).astype(np.uint32)
    _check(gpu, oracle, scene.arena, scene.tlas_offset, rays, mode, budget,
           [dict(lds_stack=k) for k in STACKS] + [dict(claim_start=5000), dict(claim_order=gpu.to_device(order), record_slab=12)])


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n,slab", [(100, 0), (8193, 5), (20000, 9)])
def test_a_scene_with_two_levels_per_node(gpu, rtx, oracle, mode, n, slab):
    _check(gpu, oracle, tiny_scene.tiny_two_depth_arena(), 0, _two_depth_rays(rtx, n, n), mode, 8192,
           [dict(record_slab=slab, lds_stack=k) for k in STACKS])


@pytest.mark.parametrize("change", [_gaps, _scales, _nan_origins])
@pytest.mark.parametrize("mode", [0, 1])
def test_unusual_nodes(gpu, oracle, instanced, mode, change):
    scene, rays = instanced
    arena = scene.arena.copy()
    change(arena, _internal_nodes(arena, scene.tlas_offset), np.random.default_rng(8))
    _check(gpu, oracle, arena, scene.tlas_offset, rays, mode, 1024, [dict(lds_stack=k) for k in STACKS])
