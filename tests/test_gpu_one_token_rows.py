"""One-token rows in a launch of the prefill kernel (decode rows of a mixed step): they stream through the decode tiles.
Every row against the float64 oracle at the edges of tiles, waves' rounds and table slices."""
import numpy as np
import pytest
import torch

import test_gpu_prefill as tp
from aicomp_amd import ops
from aicomp_amd.block_manager import StepPlan, paged_attention_step
from helpers import assert_close_attn, to_f64

pytestmark = pytest.mark.gpu

# tiles of 32 (head_dim 64: 64) tokens, four waves a round, table slices of 64 blocks
EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 513, 1023, 1024, 1025, 1153, 2049, 4200]


@pytest.mark.parametrize("dtype,kv", [(torch.bfloat16, None), (torch.float16, None), (torch.bfloat16, torch.float8_e4m3fn),
                                      (torch.float16, torch.float8_e4m3fn)])
@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 128), (4, 4, 128), (6, 2, 128), (16, 1, 128), (8, 2, 64), (4, 4, 64), (6, 2, 64),
                                      (8, 1, 64), (16, 1, 64)])
def test_one_token_rows(device, dtype, kv, hq, hkv, d):
    news = [140] + [1] * len(EDGES)                     # the chunk is long enough for two column groups, whatever the group
    c = tp.build_case(device, [70] + [n - 1 for n in EDGES], news, hq, hkv, d, dtype=dtype, kv_dtype=kv, seed=hq + d)
    want = tp.oracle(c)
    out = torch.full_like(c["q"], float("nan"))
    ops.paged_prefill_attn(out, c["q"], c["k_pool"], c["v_pool"], c["table"], c["ctx"], c["cu"], c["scale"], max_q_len=140,
                           k_scale=c["ks"], v_scale=c["vs"])
    assert_close_attn(to_f64(out), want, 1e-2, 2e-2, f"{hq}/{hkv} {d}")
    tile = ops.prefill_tile_positions(hq, hkv, d, 16, dtype, kv or dtype, 140)
    items = torch.from_numpy(ops.one_launch_items(c["ctx_list"], news, 1, tile)).to(device)
    listed = torch.full_like(c["q"], float("nan"))
    ops.paged_prefill_attn(listed, c["q"], c["k_pool"], c["v_pool"], c["table"], c["ctx"], c["cu"], c["scale"], max_q_len=140,
                           k_scale=c["ks"], v_scale=c["vs"], items=items)
    assert torch.equal(out.view(torch.int16), listed.view(torch.int16))


@pytest.mark.parametrize("d", [64, 128])
def test_scores_that_are_not_numbers(device, d):
    """A visible key that is not a number makes its row NaN, a score of -inf has no weight, as in the decode kernels."""
    c = tp.build_case(device, [70, 99, 299], [140, 1, 1], 8, 2, d, seed=d)
    c["q"][..., 3] = c["q"][..., 3].abs() + 0.5

    def run(t, key):
        k = c["k_pool"].clone()
        k[int(c["table"][2, t // 16]), :, t % 16, 3] = torch.tensor(key).to(k.dtype)
        out = torch.zeros_like(c["q"])
        ops.paged_prefill_attn(out, c["q"], k, c["v_pool"], c["table"], c["ctx"], c["cu"], c["scale"], max_q_len=140)
        return out

    for t in (0, 31, 130, 298, 299):
        out = run(t, float("nan"))
        assert torch.isnan(out[141].float()).all() and torch.isfinite(out[:141].float()).all(), t
        assert torch.equal(run(t, float("-inf")).view(torch.int16), run(t, -30000.0).view(torch.int16)), t


@pytest.mark.parametrize("kv", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("d,chunks", [(64, [200, 33]), (128, [200, 33]), (64, [9, 31]), (128, [7, 25, 16])])
def test_mixed_step_of_either_route(device, monkeypatch, kv, d, chunks):
    """More rows than a CU-round, an fp8 pool, chunks of less than a workgroup's rows: one launch against the kernels one after
    the other, pools bit for bit."""
    hq, hkv, rng, n = 16, 4, np.random.default_rng(d), len(chunks)
    news, priors = chunks + [1] * 150, [40, 0, 700][:n] + [int(x) for x in rng.integers(0, 900, 150)]
    c = tp.build_case(device, priors, news, hq, hkv, d, kv_dtype=kv, seed=d, poison=False)
    T, cu = sum(news), c["cu"].cpu().numpy()
    table = c["table"].cpu().numpy()
    pos = np.concatenate([np.arange(p, p + n) for p, n in zip(priors, news)])
    seq = np.repeat(np.arange(len(news)), news)
    slots = table[seq, pos // 16].astype(np.int64) * 16 + pos % 16
    plan = StepPlan(seq_ids=list(range(len(news))), num_prefill_seqs=n, new_lens=np.asarray(news, dtype=np.int32), max_q_len=max(chunks),
                    total_new_tokens=T, block_table=c["table"], context_lens=c["ctx"], cu_q_lens=c["cu"],
                    slot_mapping=torch.from_numpy(slots).to(device), positions=None, preempted=[],
                    host_context_lens=np.asarray(c["ctx_list"], dtype=np.int32), host_cu_q_lens=cu)
    g = torch.Generator().manual_seed(1)
    key, value = ((torch.randn(T, hkv, d, generator=g) * 0.5).to(c["q"].dtype).to(device) for _ in range(2))
    got = []
    for one in (True, False):
        plan._prefill_items = None
        if not one:
            monkeypatch.setattr(StepPlan, "ONE_LAUNCH_MAX_ROWS", 0)
        assert (plan.launch_items(c["q"], c["k_pool"]) is not None) == one
        k, v, out = c["k_pool"].clone(), c["v_pool"].clone(), torch.full_like(c["q"], float("nan"))
        paged_attention_step(plan, out, c["q"], key, value, k, v, c["scale"], c["ks"], c["vs"])
        got.append((out, k, v))
    (a, ka, va), (b, kb, vb) = got
    assert torch.equal(ka.view(torch.uint8), kb.view(torch.uint8)) and torch.equal(va.view(torch.uint8), vb.view(torch.uint8))
    t = sum(chunks) if max(chunks) >= 32 else 0               # (short chunks: another kernel alone)
    assert torch.equal(a[:t].view(torch.int16), b[:t].view(torch.int16))
    assert_close_attn(to_f64(a[t:]), to_f64(b[t:]), 1e-2, 2e-2, "rows of two kernels")
