"""The native host routes of prompt chunks and mixed steps against the calls they stand for: outputs and pools."""
import numpy as np
import pytest
import torch

import test_gpu_prefill as tp
from aicomp_amd import kv_cache, ops
from aicomp_amd.kv_cache import CachedScaledDotProductAttention
from helpers import assert_close_attn, kernels_of, to_f64

pytestmark = pytest.mark.gpu


def layouts(B, n, H, D, dtype, device, g):
    """A [B, H, n, D] tensor as attention layers hand it over: projections seen head-major, rows of a fused projection,
    head-major storage, and one whose head dimension is strided."""
    x = (torch.randn(B, n, H, D, generator=g) * 0.5).to(dtype).to(device)
    fused = torch.zeros(B, n, H + 2, D, dtype=dtype, device=device)
    fused[:, :, 1:H + 1] = x
    wide = torch.zeros(B, H, n, 2 * D, dtype=dtype, device=device)
    wide[..., ::2] = x.transpose(1, 2)
    return [x.transpose(1, 2), fused[:, :, 1:H + 1].transpose(1, 2), x.transpose(1, 2).contiguous(), wide[..., ::2]]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,hkv,group,D", [(1, 2, 4, 64), (3, 2, 4, 128), (2, 4, 1, 64)])
def test_prompt_chunks_of_the_operator(device, monkeypatch, dtype, B, hkv, group, D):
    g, hq = torch.Generator().manual_seed(B + D), hkv * group
    tol = (1e-5, 1e-5) if dtype == torch.float32 else (1e-2, 2e-2)
    for expanded in (True, False):
        for kind in range(4):
            chunks = []
            for n in (5, 2, 40):                              # the second and third continue the first
                q = layouts(B, n, hq, D, dtype, device, g)[(kind + 1) % 4]
                k, v = (layouts(B, n, hkv, D, dtype, device, g)[kind] for _ in range(2))
                if expanded:
                    k, v = k.repeat_interleave(group, 1), v.repeat_interleave(group, 1)
                chunks.append((q, k, layouts(B, n, v.shape[1], D, dtype, device, g)[kind - 1] * 0 + v if kind == 3 else v))
            got = []
            for native in (True, False):
                op = CachedScaledDotProductAttention(0, max_seq_len=64, dtype=dtype, num_kv_groups=group if expanded else None)
                op.enable()
                if not native:
                    monkeypatch.setattr(kv_cache, "_route", "torch_op")
                outs = [op(q, k, v, is_causal=True) for q, k, v in chunks]
                monkeypatch.undo()
                assert op.cache_pos == 47
                got.append((outs, op._store.k_pool.clone(), op._store.v_pool.clone()))
            (a, ka, va), (b, kb, vb) = got
            assert torch.equal(ka.view(torch.uint8), kb.view(torch.uint8)) and torch.equal(va.view(torch.uint8), vb.view(torch.uint8))
            for x, y in zip(a, b):
                assert x.shape == y.shape and x.dtype == y.dtype and x.stride() == y.stride()
                assert_close_attn(to_f64(x), to_f64(y), *tol, f"{expanded} {kind}")


@pytest.mark.parametrize("route", ["fast", "torch_op", "ctypes"])
@pytest.mark.parametrize("B,D", [(1, 64), (3, 128)])
def test_one_kv_head_repeated_by_a_view(device, monkeypatch, route, B, D):
    """One KV head repeated over the query heads without a copy, as ``repeat_kv`` does: what is kept of the view has a head
    stride of 0.  Prompt and decode against the same rows repeated by a copy."""
    hq, g, got = 8, torch.Generator().manual_seed(D), []
    monkeypatch.setattr(kv_cache, "_route", route)
    calls = [[torch.randn(B, n, h, D, generator=g).to(torch.bfloat16).to(device).transpose(1, 2) for h in (hq, 1, 1)]
             for n in (20, 3, 1, 1)]
    for copied in (False, True):
        op = CachedScaledDotProductAttention(0, max_seq_len=64, dtype=torch.bfloat16, num_kv_groups=hq)
        op.enable()
        outs = []
        for q, k, v in calls:
            n = q.shape[2]
            k, v = (x[:, :, None].expand(B, 1, hq, n, D).reshape(B, hq, n, D) for x in (k, v))
            assert k.stride(1) == 0
            if copied:
                k, v = k.contiguous(), v.contiguous()
            outs.append(op(q, k, v, is_causal=n > 1))
        got.append(outs + [op._store.k_pool, op._store.v_pool])
    for x, y in zip(*got):
        assert torch.equal(x.view(torch.int16), y.view(torch.int16))


def test_prompt_chunks_that_are_refused(device):
    op = CachedScaledDotProductAttention(0, max_seq_len=32, dtype=torch.bfloat16)
    op.enable()
    x = torch.randn(1, 4, 20, 64, device=device, dtype=torch.bfloat16)
    op(x, x, x, is_causal=True)
    with pytest.raises(RuntimeError):
        op(x, x, x, is_causal=True)                            # 40 tokens in a cache of 32
    y = torch.randn(1, 4, 5, 64, device=device)
    with pytest.raises(RuntimeError):
        op(y, y, y, is_causal=True)                            # float32 rows for a bfloat16 cache
    assert op.cache_pos == 20


@pytest.mark.parametrize("dtype,kv", [(torch.bfloat16, None), (torch.bfloat16, torch.float8_e4m3fn), (torch.float32, None)])
@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 128), (4, 4, 64), (4, 2, 256)])
@pytest.mark.parametrize("appended,lens", [(True, None), (False, None), (True, [50, 3]), (False, [50, 3])])
def test_chunks_and_rows(device, monkeypatch, dtype, kv, hq, hkv, d, appended, lens):
    news, priors = [40, 3, 1, 1, 1], [10, 0, 200, 31, 0]
    c = tp.build_case(device, priors, news, hq, hkv, d, dtype=dtype, kv_dtype=kv, seed=d)
    T, t = sum(news), 43
    rows = (torch.randn(T, 3 * hkv, d, generator=torch.Generator().manual_seed(2)) * 0.5).to(dtype).to(device)
    pos = np.concatenate([np.arange(p, p + n) for p, n in zip(priors, news)])
    table = c["table"].cpu().numpy()
    slots = torch.from_numpy(table[np.repeat(np.arange(5), news), pos // 16].astype(np.int64) * 16 + pos % 16).to(device)
    got = []
    for native in (True, False):
        k, v, out = c["k_pool"].clone(), c["v_pool"].clone(), torch.full_like(c["q"], float("nan"))
        key, value = (rows[:, :hkv], rows[:, hkv:2 * hkv]) if appended else (None, None)
        if not native:
            monkeypatch.setattr(ops, "_FAST", None)
        ops.chunks_and_rows_attn(out, c["q"], key, value, k, v, slots if appended else None, c["table"], c["ctx"], c["cu"],
                                 c["scale"], 40, 2, t, c["ks"], c["vs"], None, lens and np.asarray(lens, dtype=np.int32))
        got.append((out, k, v))
    if lens:                     # (the Python route has no kernel for few chunks)
        x, y = got[0][0], got[1][0]
        assert_close_attn(to_f64(x), to_f64(y), 1e-2, 2e-2, f"{d}")
        got = [g[1:] for g in got]
    for x, y in zip(*got):
        assert torch.equal(x.view(torch.uint8), y.view(torch.uint8))
    assert torch.isfinite(out.float()).all()


@pytest.mark.parametrize("hq,hkv,d,priors,news,longest,rows", [
    # column groups of the tile kernel: up to 144 from 640 keys on, up to 192 in pairs from 2048 (head_dim 64, one per workgroup: 64 from 900, 112 from 2048)
    (32, 8, 128, [3000, 900, 2000] + [0] * 3, [30] * 6, 3030, True), (32, 8, 128, [607] * 9, [32] * 9, 639, False),
    (32, 8, 128, [608] * 9, [32] * 9, 640, True), (16, 2, 128, [2100] + [40] * 8, [70] * 9, 2170, True),
    (16, 2, 128, [1900] + [40] * 8, [70] * 9, 1970, False), (8, 8, 128, [2036] + [100] * 20, [12] * 21, 2048, False), (16, 4, 64, [884] * 15, [16] * 15, 900, True),
    (16, 4, 64, [874] * 15, [16] * 15, 890, False), (16, 4, 64, [2032] + [100] * 24, [16] * 25, 2048, True)])
@pytest.mark.parametrize("dtype,kv", [(torch.bfloat16, None), (torch.float16, torch.float8_e4m3fn)])
def test_more_chunks_of_long_contexts(device, dtype, kv, hq, hkv, d, priors, news, longest, rows):
    c = tp.build_case(device, priors, news, hq, hkv, d, dtype=dtype, kv_dtype=kv, seed=d)
    out = torch.full_like(c["q"], float("nan"))
    names = kernels_of(lambda: ops.append_prefill_attn(
        out, c["q"], None, None, c["k_pool"], c["v_pool"], None, c["table"], c["ctx"], c["cu"], c["scale"], max(news), c["ks"],
        c["vs"], None, np.full(len(news), longest, dtype=np.int32)))
    assert any(("paged_prefill_rows" if rows else "paged_prefill_mfma") in n for n in names), names
    assert_close_attn(to_f64(out), tp.oracle(c), 1e-2, 2e-2, f"{hq}/{hkv} {d}")
