"""Batched launches of few small chunks keep to the persistent kernel with its two launches (uw_batched.hip,
few_small); the bulk path takes them where there are more chunks than resident workgroups, resolutions that
need x-slabs, extra outputs, or an octave count without a kernel of its own. Which of them ran shows in the
timed stages; meshes and records are the same on both, eager and in a graph."""
import ctypes

import numpy as np
import pytest

from test_gpu_bulk import _assert_same, _set_bulk, _snapshot, _sync
from underwaterworld_amd import params as PR

pytestmark = pytest.mark.gpu


def _stages(perlin, fn):
    from underwaterworld_amd import _lib
    L = _lib.lib()
    L.uw_profile_enable(perlin.ctx, 1)
    b = fn()
    _sync()
    ms, cnt = (ctypes.c_double * _lib.STAGE_COUNT)(), (ctypes.c_uint64 * _lib.STAGE_COUNT)()
    _lib.check(L.uw_profile_read_stages(perlin.ctx, _lib.STAGE_COUNT, ms, cnt), perlin.ctx)
    L.uw_profile_enable(perlin.ctx, 0)
    return b, [int(c) for c in cnt]


def _set(count, max_res):
    coords = [((7 * i) % 13 - 6, (5 * i) % 11 - 5, i % 3 - 2) for i in range(count)]
    return coords, [1 + (11 * i) % max_res for i in range(count)]


@pytest.mark.parametrize("octaves,max_res,count,wire,persistent", [
    (4, 12, 1, False, True), (4, 12, 24, False, True), (4, 8, 700, False, True), (6, 12, 300, False, True),
    (4, 12, 3000, False, False), (4, 13, 24, False, False), (4, 12, 24, True, False), (5, 12, 24, False, False)])
def test_few_small_chunks(octaves, max_res, count, wire, persistent):
    from underwaterworld_amd import BatchedGraph, Perlin, _lib, build_chunks_batched
    perlin = Perlin(PR.preset("chunks12", octaves=octaves), apply_tuning=False)
    coords, res = _set(count, max_res)
    opts = dict(colors=True, u16=True, collision=True) if wire else {}
    _set_bulk(perlin, 1, max_res)
    b, cnt = _stages(perlin, lambda: build_chunks_batched(perlin, coords, res, **opts))
    assert (cnt[_lib.STAGE_BULK_EMIT] == 0) == persistent
    got = _snapshot(b, count, wire)
    if not wire:
        g = BatchedGraph(perlin, coords, res)
        for _ in range(3):
            gb = g.launch()
            _sync()
            _assert_same(_snapshot(gb, count), got)
        g.close()
    _set_bulk(perlin, 0 if not persistent else max_res, max_res)  # the other path (but for max_res - 1 and below)
    other, cnt = _stages(perlin, lambda: build_chunks_batched(perlin, coords, res, **opts))
    assert (cnt[_lib.STAGE_BULK_EMIT] > 0) == persistent
    _assert_same(_snapshot(other, count, wire), got)
    t, u = b.totals(), other.totals()
    assert all(int(t[k]) == int(u[k]) for k in ("n_verts", "n_inds", "n_nonblank", "overflow"))


def test_alternating_sizes_share_a_context():
    # one context, launches going back and forth between the two kernels
    from underwaterworld_amd import Perlin, build_chunks_batched, build_chunks_plain
    perlin = Perlin(PR.preset("chunks12"))
    coords, _ = _set(2500, 12)
    ref = build_chunks_plain(perlin, coords, 12)
    _sync()
    ri = ref.info()
    for count in (24, 2500, 1, 900, 2500, 60):
        b = build_chunks_batched(perlin, coords[:count], 12)
        _sync()
        info = b.info()
        assert np.array_equal(info["n_verts"], ri["n_verts"][:count]) and np.array_equal(info["n_inds"], ri["n_inds"][:count])
        for i in range(0, count, max(1, count // 40)):
            assert all(np.array_equal(x, y) for x, y in zip(b.chunk_mesh(i, info), ref.chunk_mesh(i, ri)))
