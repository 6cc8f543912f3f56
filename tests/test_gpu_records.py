"""Records out of their slabs: row lengths around the two arrays of a slab, batch
sizes around the one-launch limit, short rays (many per chunk of records), and
scenes with 4-byte and with 8-byte slab entries.  Exact by contract, so equal to
the oracle's bit for bit."""
import os
import sys

import numpy as np
import pytest

from conftest import assert_hits_equal, assert_records_equal

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))
import tiny_scene  # noqa: E402

pytestmark = pytest.mark.gpu


def _rays(rtx, rays, n, short, seed):
    """n of the rays in a random order; `short` of them turned away (one record each) in runs."""
    rng = np.random.default_rng(seed)
    out = rays[rng.integers(0, len(rays), n)].copy()
    away = np.zeros(n, bool)
    for at in rng.integers(0, n, max(1, int(short * n) // 200)) if short else []:
        away[at:at + 200] = True
    out["org"][away] = 1e6
    out["dir"][away] = (0.0, 0.0, 1.0)
    return out


def _two_depth_rays(rtx, n, seed):
    rng = np.random.default_rng(seed)
    r = np.zeros(n, dtype=rtx.RAY_DTYPE)
    r["org"][:, :2] = rng.uniform(-1.2, 3.2, (n, 2))
    r["dir"] = (0.0, 0.0, 1.0)
    r["tmax"] = rng.choice([100.0, 4.5, 2.5], n)
    r["cull_mask"] = 0xFF
    return r


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n,short,slab", [(1, 0, 0), (255, 0.5, 31), (256, 0, 32), (257, 0, 33), (8192, 0.5, 40),
                                          (8193, 0.5, 0), (9217, 0.9, 8), (12000, 1.0, 100)])
def test_records_at_slab_and_batch_edges(gpu, rtx, oracle, instanced, mode, n, short, slab):
    scene, rays = instanced
    rays = _rays(rtx, rays, n, short, n)
    part = oracle.Partition(scene.arena, scene.tlas_offset, 1024)
    h_ref, o_ref, r_ref = oracle.trace(scene.arena, scene.tlas_offset, rays, mode=mode, partition=part)
    gpu.set_scene(scene.arena, scene.tlas_offset)
    gpu.build_treelets(1024)
    h, o, r = gpu.trace(rays, mode=mode, records=True, record_slab=slab)
    assert_hits_equal(h, h_ref, "hits")
    assert_records_equal(o, r, o_ref, r_ref, "records")


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n,slab", [(100, 0), (8192, 5), (8193, 0), (20000, 9)])
def test_records_of_a_scene_with_two_levels_per_node(gpu, rtx, oracle, mode, n, slab):
    arena = tiny_scene.tiny_two_depth_arena()
    rays = _two_depth_rays(rtx, n, n)
    part = oracle.Partition(arena, 0, 8192)
    h_ref, o_ref, r_ref = oracle.trace(arena, 0, rays, mode=mode, partition=part)
    gpu.set_scene(arena, 0)
    gpu.build_treelets(8192)
    h, o, r = gpu.trace(rays, mode=mode, records=True, record_slab=slab)
    assert_hits_equal(h, h_ref, "hits")
    assert_records_equal(o, r, o_ref, r_ref, "records")


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n", [1, 33, 1023, 1025, 9000])
@pytest.mark.parametrize("waves_per_cu", [0, 1])
def test_small_batches_by_place_and_by_counter(gpu, rtx, oracle, instanced, mode, n, waves_per_cu):
    """Waves with one ray and with eight at a time, rays taken by the wave's place (all
    resident) and from the counter (one workgroup per CU holds 8,192 of 256 CUs)."""
    scene, rays = instanced
    rays = _rays(rtx, rays, n, 0, n + 1)
    part = oracle.Partition(scene.arena, scene.tlas_offset, 1024)
    h_ref, o_ref, r_ref = oracle.trace(scene.arena, scene.tlas_offset, rays, mode=mode, partition=part)
    gpu.set_scene(scene.arena, scene.tlas_offset)
    gpu.build_treelets(1024)
    for order in (None, np.random.default_rng(n).permutation(n).astype(np.uint32)):
        claim = dict(claim_order=gpu.to_device(order)) if order is not None else {}
        rb, hb = gpu.to_device(rays), gpu.buffer(n * rtx.HIT_DTYPE.itemsize)
        assert gpu.trace_device(rb, n, hb, mode=mode, lanes_per_ray=8, waves_per_cu=waves_per_cu, **claim) == 0
        assert_hits_equal(hb.download(rtx.HIT_DTYPE, n), h_ref, "hits")
        ob, recb = gpu.buffer((n + 1) * 8), gpu.buffer(int(o_ref[-1]) * rtx.RECORD_DTYPE.itemsize)
        assert gpu.trace_device(rb, n, hb, mode=mode, records_buf=recb, record_capacity=int(o_ref[-1]), offsets_buf=ob,
                                waves_per_cu=waves_per_cu, **claim) == 0
        assert_hits_equal(hb.download(rtx.HIT_DTYPE, n), h_ref, "hits with records")
        assert_records_equal(ob.download(np.uint64, n + 1), recb.download(rtx.RECORD_DTYPE, int(o_ref[-1])), o_ref, r_ref, "records")


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n,slab", [((1 << 21) + 100, 1024), (1 << 22, 0), ((1 << 22) + 1, 0), ((1 << 23) + 1000, 0)])
def test_long_rays_in_large_batches(gpu, rtx, oracle, mode, n, slab):
    """2^31 entries hold 2,097,152 rays of 1,024-entry rows: 100 rays more are a second
    range of their own, small enough for the one-launch finish.  Rays with more records
    than a row lie in both ranges; all of them are complete.  Also one range of 4,096
    tiles and one ray more, where the tiles' sums are scanned, and two ranges of default
    rows.  Nearly all other rays miss the scene (one record each)."""
    d = rtx.workload_desc(rtx.WORKLOAD_INSTANCED_SPHERES, n_instances=600, slices=8, stacks=4, shared_blas=0, width=8,
                          height=8, seed=11, box_size=0.5)
    scene = rtx.workload_scene(d)
    long = rtx.primary_rays(d)
    gpu.set_scene(scene.arena, scene.tlas_offset)
    gpu.build_treelets(1024)
    part = oracle.Partition(scene.arena, scene.tlas_offset, 1024)
    h_ref, o_ref, r_ref = oracle.trace(scene.arena, scene.tlas_offset, long, mode=mode, partition=part)
    counts = np.diff(o_ref).astype(np.int64)
    over = np.flatnonzero(counts > 1024)
    assert len(over) >= 8
    rays = np.repeat(long[:1], n)
    rays["org"], rays["dir"] = 1e6, (0.0, 0.0, 1.0)
    # the traced rays: those with long rows, in the first range but for the last three
    at = np.concatenate([np.arange(len(over) - 3) * 7919 + 5, n - 1 - 30 * np.arange(3)[::-1]])
    rays[at] = long[over]
    h, o, r = gpu.trace(rays, mode=mode, records=True, record_slab=slab, records_per_ray=2)
    want = np.ones(n, np.uint64)
    want[at] = counts[over]
    assert np.array_equal(o, np.concatenate([[np.uint64(0)], np.cumsum(want)]))
    assert_hits_equal(h[at], h_ref[over], "hits")
    for ray, k in zip(at, over):
        assert np.array_equal(r[o[ray]:o[ray + 1]], r_ref[o_ref[k]:o_ref[k + 1]]), f"ray {ray}"
