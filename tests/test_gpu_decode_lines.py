"""Automatic decode calls above the small-call threshold that the grid schedule keeps, at its lines, append included, against
the float64 oracle."""
import numpy as np
import pytest
import torch

import test_gpu_prefill as tp
from aicomp_amd import ops
from helpers import assert_close_attn, kernels_of, to_f64

pytestmark = pytest.mark.gpu

GRID, BALANCED = "paged_decode_mfma_kernel<", "streamk_decode_kernel<"


@pytest.mark.parametrize("rows,hq,hkv,d,dtype,kv,longest,kernel,merge", [
    (64, 16, 2, 128, torch.bfloat16, None, 896, GRID, False), (64, 16, 2, 128, torch.bfloat16, None, 897, GRID, True),
    (33, 8, 8, 64, torch.float16, None, 2048, GRID, False), (130, 4, 4, 128, torch.bfloat16, None, 300, GRID, False),
    (26, 8, 8, 128, torch.bfloat16, torch.float8_e4m3fn, 1270, GRID, False), (16, 16, 8, 64, torch.bfloat16, torch.float8_e4m3fn, 3000, GRID, True),
    (64, 8, 8, 64, torch.float32, None, 1088, GRID, False), (64, 8, 8, 64, torch.float32, None, 1089, BALANCED, True),
    (60, 16, 8, 128, torch.float32, None, 640, GRID, False), (40, 16, 2, 128, torch.float32, None, 900, BALANCED, True),
    (24, 8, 8, 128, torch.bfloat16, None, 2720, GRID, True), (24, 8, 8, 128, torch.bfloat16, None, 2721, BALANCED, True)])
def test_large_calls_of_the_grid_schedule(device, rows, hq, hkv, d, dtype, kv, longest, kernel, merge):
    ops.set_small_decode_tokens(32768)                       # the library's default; restored by the suite's fixture
    rng = np.random.default_rng(rows)
    ctx = [longest] + [int(n) for n in rng.integers(1, longest + 1, rows - 1)]
    assert rows * longest > 32768
    c = tp.build_case(device, [n - 1 for n in ctx], [1] * rows, hq, hkv, d, dtype=dtype, kv_dtype=kv, seed=rows)
    want = tp.oracle(c)
    out = torch.full_like(c["q"], float("nan"))
    # the newest tokens come as arguments: what the pool holds of them is appended again
    last = torch.tensor([n - 1 for n in ctx], device=device)
    blk = c["table"].gather(1, (last // 16)[:, None].long()).squeeze(1).long()
    k0, v0 = c["k_pool"].clone(), c["v_pool"].clone()
    if kv is None:
        new = [p[blk, :, last % 16].contiguous() for p in (k0, v0)]
    else:
        new = [(p[blk, :, last % 16].float() * s[None, :, None]).to(dtype) for p, s in ((k0, c["ks"]), (v0, c["vs"]))]
    names = kernels_of(lambda: ops.paged_decode_attn(out, c["q"], c["k_pool"], c["v_pool"], c["table"], c["ctx"], c["scale"],
                                                     c["ks"], c["vs"], new_key=new[0], new_value=new[1]))
    assert any(kernel in n for n in names) and any("reduce" in n for n in names) == merge, names
    tol = (1e-5, 1e-5) if dtype == torch.float32 else (1e-2, 2e-2)
    assert_close_attn(to_f64(out), want, *tol, f"{rows} {d}")
    if kv is None:
        assert torch.equal(c["k_pool"].view(torch.uint8), k0.view(torch.uint8))
        assert torch.equal(c["v_pool"].view(torch.uint8), v0.view(torch.uint8))
