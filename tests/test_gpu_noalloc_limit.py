"""The no-allocation form takes every launch whose task records, keys, histograms, z tables and 512 bytes of
queue state fit UW_NOALLOC_SCRATCH_BYTES, to the last byte, and refuses the next."""
import numpy as np
import pytest

from test_gpu_bulk import _set_bulk
from test_zz_no_alloc import _run
from underwaterworld_amd import params as PR

pytestmark = pytest.mark.gpu

LIMIT = 32 << 20


def _need(n, octaves, max_res):
    def up(v):
        return -(-v // 256) * 256
    order = up(36 * n) + -(-n // 256) * 34 * 16 * 4
    ztab = n * (max_res + 2) * ((3 * octaves + 6) // 4 * 4) * 4
    return 512 + up(order) + up(ztab)


def _largest(octaves, max_res):
    lo, hi = 1, 1 << 20
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (mid, hi) if _need(mid, octaves, max_res) <= LIMIT else (lo, mid)
    return lo


def test_scratch_limit_to_the_last_bytes():
    from underwaterworld_amd import Perlin, _lib
    assert _lib.NOALLOC_SCRATCH_BYTES == LIMIT
    # a launch whose largest accepted chunk count comes within 512 bytes of the limit
    octaves, max_res = next((o, r) for o in range(1, 9) for r in range(1, 13) if _need(_largest(o, r), o, r) > LIMIT - 512)
    n = _largest(octaves, max_res)
    perlin = Perlin(PR.preset("chunks12", octaves=octaves), apply_tuning=False)
    _set_bulk(perlin, 0, max_res)
    coords = np.tile(np.int32([[0, 0, 9]]), (n + 300, 1))
    coords[[0, n // 2, n - 1]] = [(0, 0, -1), (1, 0, -1), (0, 1, -1)]
    vcap = icap = 1 << 20
    rc, got, _ = _run(perlin, "uw_build_chunks_batched_noalloc", coords[:n], max_res, vcap, icap)
    assert rc == _lib.UW_OK, _lib.lib().uw_last_error(perlin.ctx)
    rc, want, _ = _run(perlin, "uw_build_chunks_batched", coords[:n], max_res, vcap, icap)
    assert rc == _lib.UW_OK
    a, b = got.info()[:n], want.info()[:n]
    for f in ("flags", "n_verts", "n_inds", "n_active"):
        assert np.array_equal(a[f], b[f])
    ta, tb = got.totals(), want.totals()
    assert ta == tb and ta["overflow"] == 0
    rc, _, _ = _run(perlin, "uw_build_chunks_batched_noalloc", coords, max_res, vcap, icap)
    assert rc == _lib.UW_ERR_INVALID_ARG
