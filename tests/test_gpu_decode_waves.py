"""The grid schedule's workgroups of eight waves (partitions of more than sixteen tiles) and its whole-row
calls, around the lengths where the choice changes, against the float64 oracle at the bf16 bound."""
import numpy as np
import pytest
import torch

import test_gpu_prefill as tp
from aicomp_amd import ops
from helpers import assert_close_attn, to_f64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,kv,dtype,limit", [(128, None, torch.bfloat16, 768), (64, None, torch.float16, 1280),
                                             (128, torch.float8_e4m3fn, torch.bfloat16, 640), (64, None, torch.float32, 640),
                                             (128, None, torch.float32, 448)])
def test_rows_around_the_one_workgroup_limit(device, d, kv, dtype, limit):
    ops.set_small_decode_tokens(1 << 40)                    # the grid schedule; restored by the suite's fixture
    for longest in (limit - 255, limit - 16, limit, limit + 1):
        ctx = [longest, 1, longest - 17, 40]
        c = tp.build_case(device, [n - 1 for n in ctx], [1] * 4, 8, 2, d, dtype=dtype, kv_dtype=kv, seed=longest)
        ps = ops.decode_partition_size(4, 8, 2, d, 16, c["table"].shape[1], dtype, kv or dtype)
        assert ps == (-(-longest // 64) * 64 if longest <= limit else 256)
        got = to_f64(ops.paged_decode_attn(torch.full_like(c["q"], float("nan")), c["q"], c["k_pool"], c["v_pool"], c["table"],
                                           c["ctx"], c["scale"], c["ks"], c["vs"]))
        assert_close_attn(got, tp.oracle(c), *((1e-5, 1e-5) if dtype == torch.float32 else (1e-2, 2e-2)), f"{d} {dtype} {longest}")
        assert np.isfinite(got).all()


@pytest.mark.parametrize("rows", [32, 33])
@pytest.mark.parametrize("d,kv,dtype,longest", [(128, None, torch.bfloat16, 600), (128, torch.float8_e4m3fn, torch.bfloat16, 544),
                                               (64, None, torch.float16, 1100), (128, None, torch.float32, 288)])
def test_one_workgroup_per_cu_and_one_more_row(device, d, kv, dtype, longest, rows):
    """Partitions of more than sixteen tiles in 256 workgroups (eight waves each) and in 264 (four)."""
    ps = -(-longest // 64) * 64
    ctx = [longest - 13 * i % (longest - 1) for i in range(rows)]
    c = tp.build_case(device, [n - 1 for n in ctx], [1] * rows, 8, 8, d, dtype=dtype, kv_dtype=kv, seed=rows)
    got = to_f64(ops.paged_decode_attn(torch.full_like(c["q"], float("nan")), c["q"], c["k_pool"], c["v_pool"], c["table"],
                                       c["ctx"], c["scale"], c["ks"], c["vs"], partition_size=ps))
    assert_close_attn(got, tp.oracle(c), *((1e-5, 1e-5) if dtype == torch.float32 else (1e-2, 2e-2)), f"{d} {dtype} {rows}")


@pytest.mark.parametrize("partition", [0, 256, 448])
@pytest.mark.parametrize("d,dtype", [(128, torch.float32), (64, torch.float32), (128, torch.bfloat16), (64, torch.float16)])
def test_a_nan_score_is_a_nan_row_whatever_the_split(device, d, dtype, partition):
    """Attention over a key that is not a number has no value, as in torch; a call of one workgroup per row
    says so like one that is merged.  The other KV head's rows and the other sequence are untouched."""
    ops.set_small_decode_tokens(1 << 40)
    c = tp.build_case(device, [400, 399], [1, 1], 8, 2, d, dtype=dtype, seed=d)
    c["k_pool"][c["table"][0, 12].item(), 1, 3, 5] = float("nan")                    # token 195 of sequence 0, KV head 1
    out = ops.paged_decode_attn(torch.zeros_like(c["q"]), c["q"], c["k_pool"], c["v_pool"], c["table"], c["ctx"], c["scale"],
                                partition_size=partition)
    assert torch.isnan(out[0, 4:]).all()
    assert torch.isfinite(out[0, :4]).all() and torch.isfinite(out[1]).all() and bool(out[1].any())
