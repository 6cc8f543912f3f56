"""Node forms that decide which traversal code a scene takes: children with gaps
between them (pushed one by one instead of as a group), scales above the range of
the sign-ordered slab test, NaN origins.  Hits and records are exact by contract,
so they equal the oracle's bit for bit, with one and with eight lanes per ray."""
import numpy as np
import pytest

from conftest import assert_hits_equal, assert_records_equal

pytestmark = pytest.mark.gpu


def _internal_nodes(arena, tlas):
    """Offsets of the internal nodes reachable from the TLAS."""
    u64 = lambda o: int(arena[o:o + 8].view(np.uint64)[0])  # noqa: E731
    todo, seen = [(tlas + u64(tlas), True)], []
    while todo:
        off, top = todo.pop()
        seen.append(off)
        c = off + 64 * int(arena[off + 12:off + 16].view(np.int32)[0])
        for i in range(6):
            info = int(arena[off + 22 + i])
            size, kind = info & 3, (info >> 2) & 15
            if size and kind == 0:
                todo.append((c, top))
            elif size and top:
                h = c + u64(c + 64)
                todo.append((h + u64(h), False))
            c += 64 * size
    return seen


def _gaps(arena, nodes, rng):
    # the last child moves to the last place: a gap before it, the same memory layout
    n = 0
    for off in nodes:
        used = [i for i in range(6) if arena[off + 22 + i] & 3]
        if len(used) < 6 and rng.random() < 0.7:
            for base in (22, 28, 34, 40, 46, 52, 58):
                arena[off + base + 5] = arena[off + base + used[-1]]
            arena[off + 22 + used[-1]] = 0
            n += 1
    assert n > 10


def _scales(arena, nodes, rng):
    for off in rng.choice(nodes, 20):
        arena[off + 18 + rng.integers(0, 3)] = rng.integers(105, 127)


def _nan_origins(arena, nodes, rng):
    for off in rng.choice(nodes[1:], 5):
        arena[off:off + 4].view(np.float32)[0] = np.nan


@pytest.mark.parametrize("change", [_gaps, _scales, _nan_origins])
@pytest.mark.parametrize("mode", [0, 1])
def test_unusual_nodes_match_the_oracle(gpu, oracle, instanced, mode, change):
    scene, rays = instanced
    arena = scene.arena.copy()
    change(arena, _internal_nodes(arena, scene.tlas_offset), np.random.default_rng(4))
    part = oracle.Partition(arena, scene.tlas_offset, 1024)
    h_ref, o_ref, r_ref = oracle.trace(arena, scene.tlas_offset, rays, mode=mode, partition=part)
    gpu.set_scene(arena, scene.tlas_offset)
    gpu.build_treelets(1024)
    for stack in (4, 8, 16):
        h, o, r = gpu.trace(rays, mode=mode, records=True, lds_stack=stack)
        assert_hits_equal(h, h_ref, f"stack {stack}")
        assert_records_equal(o, r, o_ref, r_ref, f"stack {stack}")
    for lanes in (1, 8):
        assert_hits_equal(gpu.trace(rays, mode=mode, lanes_per_ray=lanes), h_ref, f"{lanes} lanes")


def _corner_rays(arena, nodes, rays, rng, far):
    """Rays through corners of child boxes, where entry and exit distances meet: world-space
    aims at TLAS children and at points of BLAS boxes, from near and from far away."""
    f32 = np.float32
    out = rays[rng.integers(0, len(rays), 4096)].copy()
    for k in range(len(out)):
        off = nodes[rng.integers(0, len(nodes))] if k % 2 else nodes[0]
        origin = arena[off:off + 12].view(f32)
        i = rng.integers(0, 6)
        corner = [origin[a] + f32(np.ldexp(float(arena[off + 28 + 12 * a + 6 * rng.integers(0, 2) + i]),
                                           int(arena[off + 18 + a:off + 19 + a].view(np.int8)[0]) - 8)) for a in range(3)]
        corner = np.array(corner, f32)
        d = rng.normal(size=3)
        kind = k % 7
        if kind < 2:  # parallel to an axis, or nearly so
            d[rng.permutation(3)[:2]] *= 0.0 if kind else 1e-6
        d = (d / np.linalg.norm(d)).astype(f32)
        o = (corner - d * f32(far * rng.uniform(0.5, 2.0))).astype(f32)
        if kind == 2:  # start on the plane
            o = corner.copy()
        out[k]["org"] = o
        out[k]["dir"] = d
        out[k]["tmin"] = 0.0
        out[k]["tmax"] = [np.inf, 4.0 * far, np.nan, -np.inf, far, 1e30, 0.0][kind]
    return out


@pytest.mark.parametrize("far", [1e-3, 1.0, 50.0, 1e5, 1e12, 1e30])
@pytest.mark.parametrize("mode", [0, 1])
def test_rays_through_box_corners_match_the_oracle(gpu, oracle, instanced, mode, far):
    scene, rays = instanced
    arena = scene.arena
    nodes = _internal_nodes(arena, scene.tlas_offset)
    rays = _corner_rays(arena, nodes, rays, np.random.default_rng(9), far)
    part = oracle.Partition(arena, scene.tlas_offset, 1024)
    h_ref, o_ref, r_ref = oracle.trace(arena, scene.tlas_offset, rays, mode=mode, partition=part)
    gpu.set_scene(arena, scene.tlas_offset)
    gpu.build_treelets(1024)
    h, o, r = gpu.trace(rays, mode=mode, records=True)
    assert_hits_equal(h, h_ref, "records")
    assert_records_equal(o, r, o_ref, r_ref, "records")
    assert_hits_equal(gpu.trace(rays, mode=mode, lanes_per_ray=1), h_ref, "hits")


def test_a_batch_reports_a_malformed_leaf_and_the_next_one_none(gpu, rtx, instanced):
    """A leaf of an unknown kind under one scene of a batch: launched directly and from a
    graph, the batch reports it each time, and a batch without that scene does not."""
    scene, rays = instanced
    bad = scene.arena.copy()
    for off in _internal_nodes(bad, scene.tlas_offset)[1:]:
        c = off + 64 * int(bad[off + 12:off + 16].view(np.int32)[0])
        for i in range(6):
            size, kind = int(bad[off + 22 + i]) & 3, (int(bad[off + 22 + i]) >> 2) & 15
            if size == 1 and kind:
                bad[c + 12] |= 1
            c += 64 * size
    n = len(rays)
    jobs = []
    for arena in (scene.arena, bad):
        sid = gpu.add_scene(arena, scene.tlas_offset)
        jobs.append((sid, gpu.to_device(rays), n, gpu.buffer(n * rtx.HIT_DTYPE.itemsize)))
    good, mixed = gpu.batch_graph(jobs[:1]), gpu.batch_graph(jobs)
    try:
        for _ in range(2):
            assert gpu.trace_batch(jobs[:1]) == 0 and good.launch()[0] == 0
            assert gpu.trace_batch(jobs) == 2 and mixed.launch()[0] == 2 and mixed.launch(2)[0] == 2
    finally:
        good.close()
        mixed.close()
