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
