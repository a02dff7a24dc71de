"""Error paths of a world update: what a caller can act on is what it gets (UW_ERR_OOM where memory is
missing), and neither the context nor the world is left in a state that a later call trips over."""
import numpy as np
import pytest

from underwaterworld_amd import params as PR
from worldcam import frustum

pytestmark = pytest.mark.gpu


def _step(world, pos, angle=0.0, reset=True):
    pos = np.float32(pos)
    bearing = np.float32([np.cos(angle), np.sin(angle), 0.05])
    return world.update(pos, bearing, frustum(pos, bearing, 55.0), frustum(pos, bearing, 90.0), sub_reset=reset)


def test_no_memory_for_a_batch_is_out_of_memory():
    # a batch of some 270,000 chunks of 32^3 cells: over 1 TB of staging
    import torch
    from underwaterworld_amd import Perlin, _lib, build_chunks_plain
    from underwaterworld_amd.world import World
    perlin = Perlin(PR.preset("reference"))
    before = build_chunks_plain(perlin, [(0, 0, -1)], 12)
    world = World(perlin, generation_dist=40, view_dist=4, min_z=-40, max_z=40, resolution=32)
    for _ in range(2):
        with pytest.raises(_lib.UwError) as e:
            _step(world, [5.0, 7.0, -3.0])
        assert e.value.code == _lib.UW_ERR_OOM
        assert world.total_count() == 0
        after = build_chunks_plain(perlin, [(0, 0, -1)], 12)  # nothing of the failure is left behind
        torch.cuda.synchronize()
        assert all(np.array_equal(x, y) for x, y in zip(before.chunk_mesh(0), after.chunk_mesh(0)))
    world.close()
