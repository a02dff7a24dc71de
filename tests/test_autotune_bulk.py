"""What the autotuner times (its timing call replaced by a synthetic cost, so no device is needed): the
persistent kernel's shape is swept and refined with the bulk path off, and the bulk threshold, every chunk
(1) among its values, is compared with the shape that won."""
import numpy as np
import pytest

from underwaterworld_amd import autotune as AT
from underwaterworld_amd import engine


@pytest.fixture
def timed(monkeypatch):
    import torch
    log = []

    def install(cost):
        def fake_time(perlin, coords, res, t, steps, stream, ref, out, label):
            log.append(dict(t, slab=list(t["slab"])))
            return cost(t)
        monkeypatch.setattr(AT, "_time_shape", fake_time)
        monkeypatch.setattr(engine, "get_batch_tuning", lambda p: dict(block=256, grid=0, max_res=32, slab=[1] * 33, bulk_min=1))
        monkeypatch.setattr(engine, "set_batch_tuning", lambda p, t: None)
        monkeypatch.setattr(torch.cuda, "current_stream", lambda: None)
        return log
    return install


def _cost(bulk):
    # the persistent kernel is best at block 192 and 6 planes of 32; a bulk launch does not see either
    def cost(t):
        if t["bulk_min"] == 1:
            return bulk
        return 1.0 + (t["block"] != 192) + 0.01 * abs(t["slab"][32] - 6) + 0.1 * (t["bulk_min"] > 1)
    return cost


@pytest.mark.parametrize("start", [None, {"block": 192, "grid": 0, "max_res": 32, "slab": AT.slabs_for_budget(28 * 1024), "bulk_min": 1}])
@pytest.mark.parametrize("bulk,chosen", [(0.5, 1), (1.5, 0)])
def test_shapes_are_timed_on_the_kernel_they_shape(timed, bulk, chosen, start):
    log = timed(_cost(bulk))
    res = [8, 12, 24, 32]
    best_ms, best = AT.tune_workload(None, np.zeros((4, 3), np.int32), res, steps=1, log=lambda *a: None, start=start)[0]
    assert (best["block"], best["slab"][32], best["bulk_min"]) == (192, 6, chosen)
    assert best_ms == (bulk if chosen else 1.0)
    thresholds = [t["bulk_min"] for t in log]
    first = next(i for i, b in enumerate(thresholds) if b)
    assert all(b == 0 for b in thresholds[:first]) and set(thresholds[first:]) >= {1, 13, 25}
    shapes = {(t["block"], tuple(t["slab"])) for t in log[first:]}
    assert len(shapes) == 1  # the thresholds are compared at the shape that won


def test_uniform_small_chunks_may_take_the_bulk_path(timed):
    log = timed(_cost(0.25))
    best = AT.tune_workload(None, np.zeros((2, 3), np.int32), [12, 12], steps=1, quick=True, log=lambda *a: None)[0][1]
    assert best["bulk_min"] == 1 and {t["bulk_min"] for t in log} == {0, 1}
