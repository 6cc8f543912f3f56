"""The device partitioner where its treelets change hands: eight lanes per
treelet for wide frontiers, one wave for instance leaves, outgrown queues and
narrow frontiers, queues in LDS or in global memory.  Checked against the
oracle's createTreelets on scenes wide enough to take each route."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# instances, slices, stacks, shared BLAS, budget
CASES = [
    (6000, 8, 4, 0, 256),      # wide frontiers that hold instance leaves
    (6000, 8, 4, 0, 1024),
    (4200, 16, 8, 0, 8192),    # subtrees that outgrow the eight-lane queue
    (4200, 16, 8, 0, 1 << 17), # one-wave queues beyond LDS
    (4200, 16, 8, 0, 1 << 20),
    (700, 16, 8, 0, 192),      # a treelet holds three nodes: many rounds
    (3, 8, 4, 0, 64 * 3),      # smallest scenes: no wide frontier
    (1500, 16, 8, 1, 512),     # one BLAS for every instance: nodes in many lists
]


@pytest.mark.parametrize("n_inst,slices,stacks,shared,budget", CASES)
def test_partition_matches_the_oracle(rtx, oracle, n_inst, slices, stacks, shared, budget):
    d = rtx.workload_desc(rtx.WORKLOAD_INSTANCED_SPHERES, n_instances=n_inst, slices=slices, stacks=stacks,
                          shared_blas=shared, width=48, height=48, seed=n_inst + budget, box_size=60.0)
    scene = rtx.workload_scene(d)
    rays = rtx.primary_rays(d)
    part = oracle.Partition(scene.arena, scene.tlas_offset, budget)
    with rtx.Context(0) as ctx:
        ctx.set_scene(scene.arena, scene.tlas_offset)
        s = ctx.build_treelets(budget)
        t = ctx.get_treelets()
        assert np.array_equal(t["roots"], part.roots)
        assert np.array_equal(t["list_offsets"], part.list_offsets)
        assert np.array_equal(t["list_nodes"], part.list_nodes)
        assert np.array_equal(t["owner"], part.owner)
        lens = np.diff(part.list_offsets.astype(np.int64))
        assert s["n_treelets"] == part.n_treelets and s["total_bytes"] == part.total_bytes
        assert s["max_treelet_nodes"] == lens.max() and s["max_treelet_bytes"] <= budget
        if not shared:  # every reachable node once: its bytes are its treelet's
            assert s["n_list_entries"] == len(np.unique(t["list_nodes"]))
        # the staged copies of the treelets hold the arena's bytes
        plain = ctx.trace(rays, mode=rtx.MODE_TREELET)
        staged = ctx.trace(rays, mode=rtx.MODE_TREELET, prefetch=rtx.PREFETCH_ALWAYS, stage_bytes=8192)
        assert ctx.prefetch_stats()["lds_hits"] > 0
        assert plain.tobytes() == staged.tobytes()


def test_lists_past_their_room_are_reported(rtx, oracle):
    """20,000 instances of 16 shared meshes: at 2 KiB the treelets' lists outgrow the room
    for them in a round of the eight-lane kernel, in the middle of a batch of rounds (at
    8 KiB in a round of the one-wave kernel).  The build reports it, and the next one, whose
    lists fit, is the oracle's."""
    rng = np.random.default_rng(5)
    builder = rtx.SceneBuilder()
    blas = [builder.add_blas(rtx.displaced_sphere(64, 32, 1.0, 0.05, seed=1 + i)) for i in range(16)]
    for i in range(20000):
        m = np.zeros((3, 4), np.float32)
        m[:, :3] = np.eye(3) * 0.5
        m[:, 3] = rng.uniform(0, 60, 3)
        builder.add_instance(int(blas[i % 16]), m, instance_id=i)
    scene = builder.finish()
    with rtx.Context(0) as ctx:
        ctx.set_scene(scene.arena, scene.tlas_offset)
        for budget in (2048, 8192):
            with pytest.raises(rtx.RtxError) as e:
                ctx.build_treelets(budget)
            assert e.value.status == 12  # out of memory
        ctx.build_treelets(256)
        part = oracle.Partition(scene.arena, scene.tlas_offset, 256)
        t = ctx.get_treelets()
        assert np.array_equal(t["roots"], part.roots)
        assert np.array_equal(t["list_offsets"], part.list_offsets)
        assert np.array_equal(t["list_nodes"], part.list_nodes)
        assert np.array_equal(t["owner"], part.owner)
