"""The coherence schedule at the sizes where its sorts change shape: around the
sort tiles (2,048 rays, 1,024 positions, 256 chunks), one to five digits of hash,
packets from one ray to more than the batch.  The schedule of the GPU's own
hashes is restated on the CPU; everything is integer, so it is equal."""
import numpy as np
import pytest

import coherence

pytestmark = pytest.mark.gpu


def _rays(rtx, n, seed, same):
    rng = np.random.default_rng(seed)
    r = np.zeros(n, rtx.RAY_DTYPE)
    d = rng.standard_normal((n, 3)).astype(np.float32)
    if same:  # a few directions only: pools of thousands of rays
        d = d[rng.integers(0, min(n, 5), n)]
    r["dir"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r["org"] = rng.uniform(0, 10, (n, 3))
    r["tmax"] = 1e30
    return r


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 2047, 2048, 2049, 4097, 40_000])
@pytest.mark.parametrize("cfg,packet", [
    (dict(hash="d", sphere_bits=1), 64), (dict(hash="d", sphere_bits=8), 64), (dict(hash="g", grid_bits=4), 32),
    (dict(hash="f", francois_bits=4), 64), (dict(hash="t", grid_bits=10), 1), (dict(hash="d", sphere_bits=4), 7),
    (dict(hash="g", grid_bits=2, sphere_bits=2), 100_000)])
def test_schedule_of_random_rays(gpu, rtx, n, cfg, packet):
    world = dict(world=rtx.COHERENCE_WORLD_GIVEN, world_min=(0.0, 0.0, 0.0), world_max=(10.0, 10.0, 10.0))
    for same in (False, True):
        rays = _rays(rtx, n, n + packet, same)
        order, hashes = gpu.coherence_order(rays, packet=packet, **cfg, **world)
        assert np.array_equal(order, coherence.packet_order_sorted(hashes, packet))
