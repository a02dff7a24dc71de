"""The persistent kernel by itself (bulk_min 0; the default sends every chunk of these sets to the bulk path):
block sizes and slab budgets against the bulk path's meshes, the interleaved queue's set-up forms, and
reservations that don't fit one packed counter. tests/test_gpu_batched.py holds the same for the default."""
import pytest

from test_gpu_batched import _assert_same, _assert_totals, _mixed_subset, _plain_by_resolution, _sync
from test_gpu_bulk import _set_bulk
from underwaterworld_amd import params as PR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("octaves", [5, 6])
@pytest.mark.parametrize("block,slab_budget", [(128, 8 * 1024), (192, 14 * 1024), (256, 20 * 1024), (512, 40 * 1024), (256, 4 * 1024)])
def test_shapes_match_the_bulk_path(block, slab_budget, octaves):
    from underwaterworld_amd import Perlin, build_chunks_batched, get_batch_tuning, set_batch_tuning
    perlin = Perlin(PR.preset("mixed", octaves=octaves))
    coords, res = _mixed_subset(64)
    t = get_batch_tuning(perlin)
    assert t["bulk_min"] == 1
    base = build_chunks_batched(perlin, coords, res)
    _sync()
    info = base.info()
    ref = {i: (info[i], *base.chunk_mesh(i, info)) for i in range(len(coords))}
    t["block"], t["bulk_min"] = block, 0
    for n in range(1, 33):
        L = n + 1
        t["slab"][n] = n if L ** 3 * 4 <= slab_budget else max(1, min(n, slab_budget // (4 * L * L) - 1))
    set_batch_tuning(perlin, t)
    b = build_chunks_batched(perlin, coords, res)
    _sync()
    _assert_same(b, ref, len(coords))
    _assert_totals(b, ref)


def test_queue_setup_forms():
    from underwaterworld_amd import Perlin, build_chunks_batched
    perlin = Perlin(PR.preset("chunks12"))
    _set_bulk(perlin, 0)
    big = [(x, y, z) for z in (-1, 0) for y in range(-50, 50) for x in range(-50, 50)]
    small = PR.grid_coords(-4, 4)
    for coords, n in ((small, 12), (big, 6), (small, 12), (big[:300], 6)):
        ref = _plain_by_resolution(perlin, coords, [n] * len(coords))
        b = build_chunks_batched(perlin, coords, [n] * len(coords))
        _sync()
        _assert_same(b, ref, len(coords))
        _assert_totals(b, ref)


def test_unpacked_reservations():
    from underwaterworld_amd import Perlin, build_chunks_batched, get_batch_tuning
    perlin = Perlin(PR.preset("mixed"))
    _set_bulk(perlin, 0)
    assert get_batch_tuning(perlin)["max_res"] == 32
    coords = [(x, y, z) for z in (-1, 0, 1) for y in range(-25, 25) for x in range(-30, 30)]
    assert 9000 * 15 * 32 ** 3 >= 2 ** 32
    ref = _plain_by_resolution(perlin, coords, [8] * len(coords))
    b = build_chunks_batched(perlin, coords, [8] * len(coords))
    _sync()
    _assert_same(b, ref, len(coords))
    _assert_totals(b, ref)
