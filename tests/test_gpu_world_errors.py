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


def _unfit(perlin):
    """A launch shape whose workgroup fits no compute unit (33^3 densities in LDS)."""
    from underwaterworld_amd import get_batch_tuning
    return dict(get_batch_tuning(perlin), bulk_min=0, max_res=32, block=512, slab=[1] + list(range(1, 33)))


def test_reported_error_does_not_reach_later_calls():
    # a batched build that HIP refuses, then calls that launch kernels of their own
    import torch
    from underwaterworld_amd import Chunk, Perlin, _lib, build_chunks_batched, get_batch_tuning, set_batch_tuning
    from underwaterworld_amd.world import World
    perlin = Perlin(PR.preset("reference"))
    good = get_batch_tuning(perlin)
    world = World(perlin)
    assert _step(world, [5.0, 7.0, -3.0]) > 0
    where = world.chunks_to_render()[0]
    want = world.get_chunk(where)
    for _ in range(2):
        set_batch_tuning(perlin, _unfit(perlin))
        with pytest.raises(_lib.UwError):
            build_chunks_batched(perlin, [where], 12)
        set_batch_tuning(perlin, good)
        got = world.get_chunk(where)
        assert np.array_equal(got.verts, want.verts) and np.array_equal(got.inds, want.inds)
    chunk = Chunk(where, resolution=12)
    chunk.build_full(perlin)
    assert np.array_equal(chunk.verts_buffer_slice(), want.verts)
    torch.cuda.synchronize()
    world.close()


def test_failed_update_gives_the_buffer_back():
    # a launch shape that HIP refuses: the update fails after its coordinates are on their way through the
    # page-locked buffer. The next holder of the buffer, another world or the same one with its
    # shape back, gets and gives its own data
    from underwaterworld_amd import Perlin, _lib, get_batch_tuning, set_batch_tuning
    from underwaterworld_amd.world import World
    perlin = Perlin(PR.preset("reference"))
    good = get_batch_tuning(perlin)
    world, other, fresh = World(perlin), World(perlin), World(perlin)
    assert _step(fresh, [5.0, 7.0, -3.0]) > 0 and _step(other, [400.0, -90.0, -3.0]) > 0
    where = [c for c in fresh.chunks_to_render()[:8]]
    there = [c for c in other.chunks_to_render()[:8]]
    want, keep = [fresh.get_chunk(c) for c in where], [other.get_chunk(c) for c in there]
    assert len(where) == 8 and len(there) == 8
    for _ in range(4):
        set_batch_tuning(perlin, _unfit(perlin))
        with pytest.raises(_lib.UwError):
            _step(world, [5.0, 7.0, -3.0])
        assert world.total_count() == 0
        for c, k in zip(there, keep):
            g = other.get_chunk(c)
            assert np.array_equal(g.verts, k.verts) and np.array_equal(g.inds, k.inds)
        set_batch_tuning(perlin, good)
    assert _step(world, [5.0, 7.0, -3.0]) > 0
    for c, w in zip(where, want):
        g = world.get_chunk(c)
        assert np.array_equal(g.verts, w.verts) and np.array_equal(g.inds, w.inds)
        assert np.array_equal(g.tri_cells, w.tri_cells) and np.array_equal(g.normals, w.normals)
    for w in (world, other, fresh):
        w.close()
