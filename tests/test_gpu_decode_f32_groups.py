"""Float32 decode with the append fused, one to five query heads per KV head (up to four share the 4 x 4 matrix
instruction): the new row's and the tiles' edges on both schedules, every row against the float64 oracle."""
import numpy as np
import pytest
import torch

import test_gpu_prefill as tp
from aicomp_amd import ops
from helpers import to_f64

pytestmark = pytest.mark.gpu


@pytest.mark.routing("balanced", "library")
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("group", [1, 2, 3, 4, 5])
def test_groups_of_heads(device, decode_routing, group, d):
    ctx = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 300]
    c = tp.build_case(device, [n - 1 for n in ctx], [1] * len(ctx), 2 * group, 2, d, dtype=torch.float32, seed=group + d,
                      poison="all")
    want = tp.oracle(c)
    # the newest row moves from the pools to the call's arguments
    new_k, new_v = (torch.empty(len(ctx), 2, d, device=device) for _ in range(2))
    kp, vp = c["k_pool"].clone(), c["v_pool"].clone()
    for s, n in enumerate(ctx):
        blk, off = int(c["table"][s, (n - 1) // 16]), (n - 1) % 16
        new_k[s], new_v[s] = c["k_pool"][blk, :, off], c["v_pool"][blk, :, off]
        kp[blk, :, off], vp[blk, :, off] = float("nan"), float("inf")
    for partition in (0, 64, 128):
        k, v, out = kp.clone(), vp.clone(), torch.full_like(c["q"], float("nan"))
        ops.paged_decode_attn(out, c["q"], k, v, c["table"], c["ctx"], c["scale"], partition_size=partition, new_key=new_k,
                              new_value=new_v)
        err = np.abs(to_f64(out) - want).max()
        assert err <= 1e-5, (partition, err)                # float32 sums of at most 300 keys of N(0, 1/4)
        assert torch.equal(k.view(torch.int32), c["k_pool"].view(torch.int32))
        assert torch.equal(v.view(torch.int32), c["v_pool"].view(torch.int32))
