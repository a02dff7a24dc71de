"""Calls on a device whose memory is taken: what the context keeps for later uses is given up before a call
fails for want of memory. The memory is taken by plain allocations, all but a few dozen MiB, and given back."""
import contextlib
import ctypes

import numpy as np
import pytest

from test_gpu_world_errors import _step
from underwaterworld_amd import params as PR

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@contextlib.contextmanager
def _memory_left(mib):
    """About `mib` MiB of device memory are left free inside."""
    import torch
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    spare = torch.empty(mib * MIB, dtype=torch.uint8, device="cuda")
    held, size = [], 32 << 30
    while size >= 4 * MIB:
        try:
            held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
        except torch.cuda.OutOfMemoryError:
            size //= 2
    del spare
    torch.cuda.empty_cache()
    try:
        yield
    finally:
        held.clear()
        torch.cuda.synchronize()
        torch.cuda.empty_cache()


def test_kept_blocks_make_room():
    import torch
    from underwaterworld_amd import Perlin, _lib, build_chunks_plain
    from underwaterworld_amd.engine import _alloc_out, _mesh_out, _stream_ptr
    from underwaterworld_amd.world import World
    perlin = Perlin(PR.preset("reference"))
    few = build_chunks_plain(perlin, [(0, 0, -1)], 12)  # (the kernels are loaded while there is memory)
    world = World(perlin)
    assert _step(world, [5.0, 7.0, -3.0]) > 250
    world.close()  # over 100 MB stay with the context
    count = 8192
    coords = torch.as_tensor(np.tile(np.int32([[0, 0, 9]]), (count, 1)), device="cuda")
    coords[0] = torch.tensor([0, 0, -1], dtype=torch.int32)
    verts, inds, info, totals = _alloc_out(count, 20000, 60000, "cuda")
    out = _mesh_out(verts, inds, info, totals, 20000, 60000)
    with _memory_left(24):  # its scratch takes about 95 MB
        _lib.check(_lib.lib().uw_build_chunks_plain(perlin.ctx, ctypes.c_void_p(coords.data_ptr()), count, 12, ctypes.byref(out),
                                                    None, _stream_ptr(None)), perlin.ctx)
        torch.cuda.synchronize()
    v, ix = few.chunk_mesh(0)
    assert np.array_equal(verts[:len(v)].cpu().numpy(), v) and np.array_equal(inds[:len(ix)].cpu().numpy().view(np.uint32), ix)


@pytest.mark.parametrize("octaves,n,count,left", [(4, 12, 8192, 64), (6, 24, 3000, 400)])
def test_batched_without_room_for_the_bulk_scratch(octaves, n, count, left):
    # scratch of about 110 and 480 MB that the bulk path would take; the persistent kernel needs none for
    # chunks built in one pass and about 150 MB for those in x-slabs. Graphs own theirs, in the same way
    import torch
    from underwaterworld_amd import BatchedGraph, Perlin, build_chunks_batched
    perlin = Perlin(PR.preset("chunks12" if octaves == 4 else "mixed", octaves=octaves))
    coords = torch.as_tensor(np.tile(np.int32([[0, 0, 9]]), (count, 1)), device="cuda")
    coords[:4] = torch.tensor([[0, 0, -1], [3, 1, -1], [0, 0, 0], [1, 2, 0]], dtype=torch.int32)
    res = torch.full((count,), n, dtype=torch.int32, device="cuda")
    few = build_chunks_batched(Perlin(perlin.params), coords[:4], n)
    caps = dict(vert_cap=60000, ind_cap=200000)
    other = Perlin(perlin.params, apply_tuning=False)
    from test_gpu_bulk import _set_bulk
    _set_bulk(other, 0)  # (the persistent kernel is loaded while there is memory)
    build_chunks_batched(other, coords[:4], n)
    torch.cuda.synchronize()
    with _memory_left(left):
        b = build_chunks_batched(perlin, coords, res, **caps)
        g = BatchedGraph(perlin, coords, res, **caps)
        gb = g.launch()
        torch.cuda.synchronize()
    again = build_chunks_batched(perlin, coords, res, **caps)
    torch.cuda.synchronize()
    want = few.info()
    for got in (b, gb, again):
        info = got.info()
        assert got.totals()["overflow"] == 0 and not info["n_inds"][4:].any()
        for i in range(4):
            assert tuple(info[i])[:4] == tuple(want[i])[:4]
            assert all(np.array_equal(x, y) for x, y in zip(got.chunk_mesh(i, info), few.chunk_mesh(i, want)))
    g.close()
