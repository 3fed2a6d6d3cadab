"""Split rows of the grid schedule whose partitions turn with the row (numbers of partitions divisible by four) and those
beside them, append included, against the float64 oracle."""
import pytest
import torch

import test_gpu_prefill as tp
from aicomp_amd import ops
from helpers import assert_close_attn, kernels_of, to_f64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,kv,d", [(torch.bfloat16, None, 128), (torch.float16, torch.float8_e4m3fn, 64), (torch.float32, None, 64)])
@pytest.mark.parametrize("rows,hkv,parts", [(1, 2, 4), (5, 1, 4), (21, 2, 8), (9, 2, 12), (37, 1, 16), (6, 2, 20), (7, 2, 6)])
def test_every_partition_of_every_row(device, dtype, kv, d, rows, hkv, parts):
    longest = 64 * parts
    ctx = [longest if s % 4 == 0 else 1 + (97 * s) % longest for s in range(rows)]
    c = tp.build_case(device, [n - 1 for n in ctx], [1] * rows, 4 * hkv, hkv, d, dtype=dtype, kv_dtype=kv, seed=rows + parts)
    last = torch.tensor([n - 1 for n in ctx], device=device)
    blk = c["table"].gather(1, (last // 16)[:, None].long()).squeeze(1).long()
    k0, v0 = c["k_pool"].clone(), c["v_pool"].clone()
    new = [p[blk, :, last % 16].float() * (1 if s is None else s[None, :, None]) for p, s in ((k0, c["ks"]), (v0, c["vs"]))]
    out = torch.full_like(c["q"], float("nan"))
    names = kernels_of(lambda: ops.paged_decode_attn(out, c["q"], c["k_pool"], c["v_pool"], c["table"], c["ctx"], c["scale"], c["ks"],
                                                     c["vs"], partition_size=64, new_key=new[0].to(dtype), new_value=new[1].to(dtype)))
    assert any("paged_decode_mfma_kernel<" in n for n in names) and any("split_reduce" in n for n in names), names
    assert_close_attn(to_f64(out), tp.oracle(c), *((1e-5, 1e-5) if dtype == torch.float32 else (1e-2, 2e-2)), f"{rows} {parts}")
    if kv is None:
        assert torch.equal(c["k_pool"].view(torch.uint8), k0.view(torch.uint8))
        assert torch.equal(c["v_pool"].view(torch.uint8), v0.view(torch.uint8))
