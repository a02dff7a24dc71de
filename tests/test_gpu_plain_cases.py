"""Cube cases of every cell beside a plain build (chunk.rs:155-162): where rows are written in words (cells
per axis a multiple of four, buffer on a word) and in bytes, at one row segment and two, for chunks with and
without surface, in launches of few and of many workgroups; and a launch of more than 2^32 cells."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from underwaterworld_amd import params as PR

pytestmark = pytest.mark.gpu

COORDS = [(0, 0, -1), (3, 1, -1), (0, 0, 6), (-2, 4, -1), (1, 1, -9), (2, -1, 0)]


def _build(perlin, coords, n, cases):
    """A build that only reports sizes (no room for meshes) and writes the cases at address `cases`."""
    import torch
    from underwaterworld_amd import _lib
    from underwaterworld_amd.engine import _alloc_out, _coords_tensor, _mesh_out, _stream_ptr
    dev = torch.device("cuda", 0)
    ct = _coords_tensor(coords, dev)
    verts, inds, info, totals = _alloc_out(len(ct), 0, 0, dev)
    out = _mesh_out(verts, inds, info, totals, 0, 0)
    _lib.check(_lib.lib().uw_build_chunks_plain(perlin.ctx, ctypes.c_void_p(ct.data_ptr()), len(ct), n, ctypes.byref(out),
                                                ctypes.c_void_p(cases), _stream_ptr(None)), perlin.ctx)
    torch.cuda.synchronize()


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n", [1, 3, 4, 12, 31, 32, 33, 36, 64])
def test_cases_match_oracle(n, shift):
    import torch
    from underwaterworld_amd import Perlin, sample_density
    p = PR.preset("mixed", octaves=3)
    perlin = Perlin(p)
    dens, _ = sample_density(perlin, COORDS, n)
    want = [O.mesh_ref(p, c, n, d)["cases"] for c, d in zip(COORDS, dens.cpu().numpy())]
    count = 6 if n > 12 else 1200
    buf = torch.full((count * n ** 3 + 64,), 77, dtype=torch.uint8, device="cuda")
    _build(perlin, [COORDS[i % 6] for i in range(count)], n, buf.data_ptr() + shift)
    got = buf.cpu().numpy()
    assert (got[:shift] == 77).all() and (got[shift + count * n ** 3:] == 77).all()
    assert np.array_equal(got[shift:shift + count * n ** 3].reshape(count, -1), np.array([want[i % 6] for i in range(count)]))


def test_more_cells_than_32_bits():
    import torch
    from underwaterworld_amd import Perlin
    n, count = 64, 16390  # 4.3e9 cells
    assert count * n ** 3 > 1 << 32
    perlin = Perlin(PR.preset("mixed", octaves=1))
    few = torch.empty(len(COORDS) * n ** 3, dtype=torch.uint8, device="cuda")
    _build(perlin, COORDS, n, few.data_ptr())
    coords = np.tile(np.int32([[0, 0, 7]]), (count, 1))
    coords[:6], coords[-6:] = COORDS, COORDS
    cases = torch.full((count * n ** 3,), 77, dtype=torch.uint8, device="cuda")
    _build(perlin, coords, n, cases.data_ptr())
    assert torch.equal(cases[:few.numel()], few) and torch.equal(cases[-few.numel():], few)
    assert int(cases[few.numel():-few.numel()].max()) == 0
    del cases
    torch.cuda.empty_cache()
