"""What the native launch path refuses before it launches anything, on tensors in host memory: no GPU is needed."""
import dataclasses

import numpy as np
import pytest
import torch

from mlora import AdapterPool, _ext, ops


def _pool(n_slots=4):
    pool = AdapterPool(1, {"p": (64, 64)}, n_slots, n_slots * 2, page_rows=8, max_rank=16, device="cpu")
    for s in range(n_slots):
        pool.allocate(s, 16, 1.0)
    return pool


def _plan(T, pool):
    i32 = dict(dtype=torch.int32)
    segs = min(T, pool.n_slots)
    return ops.DecodePlan(torch.zeros(T, **i32), 1, torch.zeros(T, **i32), *(torch.zeros(segs, **i32) for _ in range(3)),
                          *(torch.zeros(T, **i32) for _ in range(3)), torch.zeros(_ext.CNT_WORDS, **i32),
                          torch.zeros((_ext.work_cap(T), _ext.WORK_WORDS), **i32), torch.zeros((T, pool.max_pages), **i32),
                          torch.zeros(T, **i32), torch.zeros(T))


BUFFERS = ["perm", "seg_start", "seg_len", "seg_adapter", "chunk_start", "chunk_len", "chunk_adapter", "counters", "work",
           "row_off", "tok_rank", "tok_scale"]


@pytest.mark.parametrize("name", BUFFERS)
def test_gather_refuses_a_plan_whose_buffers_are_too_small(name):
    """Every buffer one value short of what the gather kernel writes for this batch and pool."""
    pool = _pool()
    plan = _plan(9, pool)
    setattr(plan, name, getattr(plan, name).reshape(-1)[:-1].contiguous())
    with pytest.raises(ValueError, match=name):
        _ext.host().gather(pool, plan, torch.zeros(9, dtype=torch.int32), 1)


def test_gather_refuses_a_larger_pool_and_other_buffers():
    plan = _plan(9, _pool(4))
    with pytest.raises(ValueError, match="seg_start"):           # nine tokens, up to eight adapters
        _ext.host().gather(_pool(8), plan, torch.zeros(9, dtype=torch.int32), 1)
    for name, other in (("perm", torch.zeros(9, dtype=torch.int64)), ("tok_scale", torch.zeros(9, dtype=torch.int32)),
                        ("work", torch.zeros(_ext.WORK_WORDS, 16, dtype=torch.int32).t())):
        with pytest.raises(ValueError, match=name):
            _ext.host().gather(_pool(), dataclasses.replace(_plan(9, _pool()), **{name: other}), torch.zeros(9, dtype=torch.int32), 1)
    with pytest.raises(ValueError, match="device tensors"):      # the buffers fit: what is left to refuse is host memory
        _ext.host().gather(_pool(), _plan(9, _pool()), torch.zeros(9, dtype=torch.int32), 1)


@pytest.mark.parametrize("weights, error", [
    ([torch.zeros(2, 1, 8, 16), torch.zeros(2, 1, 24, 8)], "device tensors"),          # the input and the pool are in host memory
    ([torch.zeros(2, 1, 8, 16)], "one wa and wb each"),
    ([], "one wa and wb each"),
])
def test_reference_layout_deltas_check_their_tensors(weights, error):
    plan = ops.RefDecodePlan(torch.zeros(3, dtype=torch.int64), 1, 2, 1, 8, torch.zeros(16, dtype=torch.uint8))
    with pytest.raises(ValueError, match=error):
        _ext.host().deltas_ref(plan, torch.zeros(3, 16), weights, 0, 3, 2, 1, 8)
