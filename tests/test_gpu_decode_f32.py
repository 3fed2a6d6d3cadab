"""Float32 decode on the float32 matrix instruction, at the edges of its tiles, against the float64 oracle.

Tolerance: with |q . k| / sqrt(D) of a few units and |v| <= 2.5 every product and sum is float32; the
scores carry at most D roundings of 2^-24 relative to sum |q k| (about 1e-6), the output the same
relative error again: 1e-5 absolute covers both with a factor of four to spare.
"""
import numpy as np
import pytest
import torch

import test_gpu_prefill as tp
from aicomp_amd import ops
from helpers import to_f64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("group", [1, 3, 4, 8, 16])
@pytest.mark.parametrize("schedule", ["balanced", "grid"])
def test_f32_decode_tile_edges(device, d, group, schedule):
    """Context lengths around tiles of 16 and 32 tokens, the one-workgroup limit and several waves;
    non-finite pool contents beyond every context; append fused and unfused; both schedules."""
    ops.set_small_decode_tokens(0 if schedule == "balanced" else 1 << 40)     # restored by the suite's fixture
    hkv = 2
    ctx = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 129, 300, 511]
    c = tp.build_case(device, [n - 1 for n in ctx], [1] * len(ctx), group * hkv, hkv, d, dtype=torch.float32, seed=d + group,
                      poison="all")
    want = tp.oracle(c)
    args = (c["table"], c["ctx"], c["scale"])
    got = to_f64(ops.paged_decode_attn(torch.full_like(c["q"], float("nan")), c["q"], c["k_pool"], c["v_pool"], *args))
    assert np.isfinite(got).all() and np.abs(got - want).max() <= 1e-5
    # the newest token arrives with the call: same pools, same output as append then attend
    kp, vp = c["k_pool"].clone(), c["v_pool"].clone()
    rows = [int(c["table"][s, (n - 1) // 16]) for s, n in enumerate(ctx)]
    at = [(n - 1) % 16 for n in ctx]
    nk, nv = kp[rows, :, at].clone(), vp[rows, :, at].clone()
    kp[rows, :, at], vp[rows, :, at] = float("nan"), float("nan")
    fused = ops.paged_decode_attn(torch.empty_like(c["q"]), c["q"], kp, vp, *args, new_key=nk, new_value=nv)
    assert np.array_equal(to_f64(fused), got)
    bits = lambda t: t.view(torch.int32)
    assert torch.equal(bits(kp), bits(c["k_pool"])) and torch.equal(bits(vp), bits(c["v_pool"]))
