"""Kernel timing of batched builds (uw_profile_read, uw_profile_read_stages): stage 0, the one that
uw_profile_read returns, is recorded once per build whichever kernels it takes, and the stages of a build
don't overlap."""
import ctypes

import pytest

from test_gpu_bulk import _set_bulk
from underwaterworld_amd import params as PR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bulk_min,rows,emit", [(1, 1, 1), (0, 0, 0), (17, 1, 1)])
def test_stage_zero_of_batched_builds(bulk_min, rows, emit):
    import torch
    from underwaterworld_amd import Perlin, _lib, build_chunks_batched
    L = _lib.lib()
    perlin = Perlin(PR.preset("mixed"))
    if bulk_min != 1:
        _set_bulk(perlin, bulk_min)
    coords, res = PR.mixed_workload(8192, 7)
    coords, res, calls = coords[:600], res[:600], 5
    build_chunks_batched(perlin, coords, res)
    torch.cuda.synchronize()
    L.uw_profile_enable(perlin.ctx, 1)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(calls):
        build_chunks_batched(perlin, coords, res)
    e1.record()
    torch.cuda.synchronize()
    n = _lib.STAGE_COUNT
    ms, cnt = (ctypes.c_double * n)(), (ctypes.c_uint64 * n)()
    _lib.check(L.uw_profile_read_stages(perlin.ctx, n, ms, cnt), perlin.ctx)
    assert cnt[_lib.STAGE_DOMINANT] == calls and ms[_lib.STAGE_DOMINANT] > 0.0
    assert cnt[_lib.STAGE_BATCH_SETUP] == calls
    assert cnt[_lib.STAGE_BULK_FRONT] == calls * rows and cnt[_lib.STAGE_BULK_EMIT] == calls * emit
    assert sum(ms) <= e0.elapsed_time(e1)
    for _ in range(calls):
        build_chunks_batched(perlin, coords, res)
    total, launches = ctypes.c_double(), ctypes.c_uint64()
    _lib.check(L.uw_profile_read(perlin.ctx, ctypes.byref(total), ctypes.byref(launches)), perlin.ctx)
    L.uw_profile_enable(perlin.ctx, 0)
    assert launches.value == calls and total.value > 0.0
