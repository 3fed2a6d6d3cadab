"""The natively planned decode step against the planner's own numpy code: the same plans, field by field, and the same
state after every step, over random arrivals, finishes and preemptions."""
import random

import numpy as np
import pytest
import torch

import aicomp_amd.block_manager as bm

ARRAYS = ("new_lens", "host_block_table", "host_context_lens", "host_cu_q_lens", "host_slot_mapping", "host_positions",
          "block_table", "context_lens", "cu_q_lens", "slot_mapping", "positions")
DEVICE = ARRAYS[6:]


def _plans_equal(monkeypatch, seed, device):
    native, rng = bm._FAST, random.Random(seed)
    blocks, budget = rng.choice([(40, 60), (25, 4), (200, 60)])
    pair = [bm.StepPlanner(blocks, 16, max_seqs=6, max_seq_len=200 if seed % 2 else 130,
                           max_num_batched_tokens=budget, prefill_chunk=32, device=device) for _ in range(2)]
    kept = []                                                # the last three plans

    def step(p, fast):
        monkeypatch.setattr(bm, "_FAST", native if fast else None)
        try:
            plan = p.schedule()
        except ValueError as e:
            plan = str(e)
        return plan, p.completed()

    for i in range(60):
        if rng.random() < 0.2:
            n, m = rng.randint(1, 120), rng.choice([None, 0, 1, 5, 40])
            for p in pair:
                try:
                    p.add_request(i, n, m)
                except ValueError:
                    pass
        (x, done), (y, done_y) = step(pair[0], True), step(pair[1], False)
        assert type(x) is type(y) and done == done_y
        if isinstance(x, str):
            assert x == y
            break
        if x is not None:
            for f in ("seq_ids", "num_prefill_seqs", "max_q_len", "total_new_tokens", "preempted"):
                assert getattr(x, f) == getattr(y, f), f
            for f in ARRAYS:
                u, v = getattr(x, f), getattr(y, f)
                assert u.dtype == v.dtype and u.shape == v.shape and (u == v).all(), f
            # on the device what the host has, also three plans later
            kept = (kept + [x])[-3:]
            for plan in kept:
                for f in DEVICE:
                    t = getattr(plan, f)
                    assert t.device.type == torch.device(device).type
                    if t.is_cuda:
                        assert (t.cpu().numpy() == getattr(plan, "host_" + f)).all(), f
        for p in pair:
            for sid in done:
                p.finish(sid)
        a, b = pair
        assert a.alloc._top == b.alloc._top and (a.alloc._free == b.alloc._free).all()
        assert (a.alloc._owned == b.alloc._owned).all()
        assert all(np.array_equal(u, v) for u, v in zip(a._row_state + (a._tab,), b._row_state + (b._tab,)))


@pytest.mark.skipif(bm._FAST is None, reason="csrc/fast_call.cpp is not built")
@pytest.mark.parametrize("seed", range(40))
def test_plans_equal_the_numpy_planner(monkeypatch, seed):
    _plans_equal(monkeypatch, seed, "cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("seed", range(8))
def test_plans_reach_the_device(monkeypatch, device, seed):
    """The native upload: staged in pinned memory, copied asynchronously, a ring of buffers."""
    _plans_equal(monkeypatch, seed, "cuda")
