"""A step of prompt chunks alone (append and attention in one call) on either side of the line below which a chunk's keys
are split between waves: every row against the float64 oracle, the pools bit for bit, the same bits with an item list."""
import numpy as np
import pytest
import torch

import test_gpu_prefill as tp
from aicomp_amd import ops
from helpers import assert_close_attn, kernels_of, to_f64

pytestmark = pytest.mark.gpu

ROWS, TILES = "paged_prefill_rows_kernel<", "paged_prefill_mfma_kernel<"
LONG = 1 << 20                       # a longest context that makes few chunks take the kernel that splits their keys


def lens(n, longest=LONG):
    return np.full(n, longest, dtype=np.int32)


# chunk lengths and priors at the edges of 16-row workgroups, 32- and 64-token tiles and the waves' rounds
CHUNKS = [([0], [1]), ([0], [17]), ([31], [33]), ([0, 63, 64, 65], [64, 1, 2, 15]), ([127, 128, 129], [16, 17, 31]),
          ([500, 0, 255, 257], [40, 129, 3, 65]), ([1000], [48]), ([2049, 7], [5, 20])]


@pytest.mark.parametrize("dtype,kv", [(torch.bfloat16, None), (torch.float16, None), (torch.bfloat16, torch.float8_e4m3fn)])
@pytest.mark.parametrize("hq,hkv,d", [(4, 4, 128), (8, 2, 128), (16, 2, 64), (6, 2, 64), (16, 1, 64), (16, 1, 128)])
def test_chunks_alone(device, dtype, kv, hq, hkv, d):
    for i, (priors, news) in enumerate(CHUNKS):
        c = tp.build_case(device, priors, news, hq, hkv, d, dtype=dtype, kv_dtype=kv, seed=i + d)
        want = tp.oracle(c)
        outs = []
        for listed in (False, True):
            items = None
            tile = ops.prefill_tile_positions(hq, hkv, d, 16, dtype, kv or dtype, max(news))
            if listed and tile:
                group = hq // hkv
                items = torch.from_numpy(ops.prefill_items(np.asarray(c["ctx_list"], dtype=np.int32), np.asarray(news, dtype=np.int32), tile,
                                                           hq // (group if 16 % group == 0 else 1), 256)).to(device)
            out = torch.full_like(c["q"], float("nan"))
            names = kernels_of(lambda: ops.append_prefill_attn(
                out, c["q"], None, None, c["k_pool"], c["v_pool"], None, c["table"], c["ctx"], c["cu"], c["scale"], max(news),
                c["ks"], c["vs"], items, lens(len(news))))
            # (16 heads of 64, and more than 32 workgroups of the other kernel at D 64)
            which = TILES if d == 64 and (hq // hkv == 16 or (hq, max(news)) == (16, 129)) else ROWS
            assert any(which in n for n in names), names
            outs.append(out)
            assert_close_attn(to_f64(out), want, 1e-2, 2e-2, f"{hq}/{hkv} {d} {priors} {news}")
        assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.parametrize("dtype,kv", [(torch.bfloat16, None), (torch.float16, torch.float8_e4m3fn), (torch.float32, None)])
@pytest.mark.parametrize("hq", [4, 48])
def test_append_and_attention_in_one_call(device, dtype, kv, hq):
    """The new rows come as arguments, strided; 48 heads are beyond the line."""
    priors, news, hkv, d = [5, 200], [70, 33], hq // 2, 64
    c = tp.build_case(device, priors, news, hq, hkv, d, dtype=dtype, kv_dtype=kv, seed=hq)
    want_k, want_v, T = c["k_pool"].clone(), c["v_pool"].clone(), sum(news)
    rows = (torch.randn(T, 2 * hkv, d, generator=torch.Generator().manual_seed(1)) * 0.5).to(dtype).to(device)
    key, value = rows[:, :hkv], rows[:, hkv:]
    slots = torch.cat([c["table"][s, t // 16].long() * 16 + t % 16 for s, (p, n) in enumerate(zip(priors, news))
                       for t in [torch.arange(p, p + n, device=device)]])
    ops.kv_append(key, value, want_k, want_v, slots, c["ks"], c["vs"])
    out = torch.full_like(c["q"], float("nan"))
    ops.append_prefill_attn(out, c["q"], key, value, c["k_pool"], c["v_pool"], slots, c["table"], c["ctx"], c["cu"],
                            c["scale"], max(news), c["ks"], c["vs"])
    assert torch.equal(c["k_pool"].view(torch.uint8), want_k.view(torch.uint8))
    assert torch.equal(c["v_pool"].view(torch.uint8), want_v.view(torch.uint8))
    tol = (1e-5, 1e-5) if dtype == torch.float32 else (1e-2, 2e-2)
    assert_close_attn(to_f64(out), tp.oracle(c), *tol, f"{dtype} {hq}")


def test_chunks_alone_zero_rows_and_junk_pairs(device):
    """A context shorter than its chunk gives zero rows; pairs of the list that name nothing are skipped."""
    c = tp.build_case(device, [0, 10], [40, 20], 4, 4, 128, seed=3)
    c["ctx"][0] = 39
    for items in (None, torch.tensor([[0, 0], [-1, 0], [1, 0], [7, 0], [1, 90], [0, -2], [1, 2 ** 30]], dtype=torch.int32, device=device)):
        out = torch.full_like(c["q"], float("nan"))
        ops.append_prefill_attn(out, c["q"], None, None, c["k_pool"], c["v_pool"], None, c["table"], c["ctx"], c["cu"],
                                c["scale"], 40, None, None, items, lens(2))
        assert (out[:40] == 0).all() and torch.isfinite(out.float()).all()
        want = tp.oracle(dict(c, ctx_list=[40, 30]))[40:]
        assert_close_attn(to_f64(out[40:]), want, 1e-2, 2e-2, "second chunk")


@pytest.mark.parametrize("dtype,kv", [(torch.bfloat16, None), (torch.float16, None), (torch.float16, torch.float8_e4m3fn)])
@pytest.mark.parametrize("hq,hkv,d", [(4, 4, 64), (8, 2, 64), (6, 2, 64), (16, 2, 64), (8, 2, 128)])
def test_keys_a_row_does_not_see(device, dtype, kv, hq, hkv, d):
    """A later token's key that is not finite leaves the rows before it as they are, bit for bit; a visible key whose score
    is -inf has weight 0, like one whose exponential underflows."""
    c = tp.build_case(device, [2], [41], hq, hkv, d, dtype=dtype, kv_dtype=kv, seed=d + hq)
    c["q"][..., 7] = c["q"][..., 7].abs() + 0.5

    def run(t=None, key=None):
        k = c["k_pool"].clone()
        if t is not None:
            rows = k[int(c["table"][0, (2 + t) // 16]), :, (2 + t) % 16]
            rows[:, 7] = torch.tensor(key).to(k.dtype)
            if kv is not None:
                rows[:, 7] = torch.tensor(float("nan")).to(k.dtype)      # (e4m3 has no infinities)
        out = torch.full_like(c["q"], float("nan"))
        ops.append_prefill_attn(out, c["q"], None, None, k, c["v_pool"], None, c["table"], c["ctx"], c["cu"], c["scale"], 41,
                                c["ks"], c["vs"], None, lens(1))
        return out.view(torch.int16)

    clean = run()
    assert torch.isfinite(clean.view(dtype)).all()
    for t in (1, 2, 13, 14, 29, 30, 31, 40):
        for key in (float("inf"), float("nan"), float("-inf")):
            assert torch.equal(run(t, key)[:t], clean[:t]), (t, key)
        if kv is None:
            assert torch.equal(run(t, float("-inf")), run(t, -30000.0)), t


@pytest.mark.parametrize("hq,hkv,d,priors,news,longest,kernel", [
    # one column group of the other kernel: from 256 keys on (head_dim 64: 192)
    (8, 8, 128, [0] * 4, [24] * 4, 255, TILES), (8, 8, 128, [232] * 4, [24] * 4, 256, ROWS),
    (8, 8, 64, [91], [100], 191, TILES), (8, 8, 64, [92], [100], 192, ROWS),
    # two: at once, up to 32 workgroups, of one chunk up to 64 (head_dim 64: up to 32 column groups, beyond that from 600 keys on)
    (32, 8, 128, [0, 0], [46, 46], 46, ROWS), (16, 2, 64, [0] * 4, [24] * 4, 24, ROWS),
    (32, 8, 128, [0], [200], 200, ROWS),
    (32, 8, 64, [499], [100], 599, TILES), (32, 8, 64, [500], [100], 600, ROWS),
    # 33 to 64 workgroups, of four waves each here; the block table is read again every 64 entries
    (32, 8, 128, [0] * 4, [46] * 4, 46, TILES), (32, 8, 128, [1054, 2100, 0, 700], [46, 40, 33, 46], 2140, ROWS),
    (32, 8, 128, [1200], [200], 1400, ROWS), (16, 2, 64, [700] * 8, [46] * 8, 746, TILES), (64, 8, 128, [0], [200], LONG, TILES),
    # beyond both
    (64, 8, 64, [700] * 4, [46] * 4, 746, TILES)])
@pytest.mark.parametrize("dtype,kv", [(torch.bfloat16, None), (torch.float16, torch.float8_e4m3fn)])
def test_lines(device, dtype, kv, hq, hkv, d, priors, news, longest, kernel):
    """Which kernel a step of chunks takes, by what the host knows of its contexts; either is right."""
    c = tp.build_case(device, priors, news, hq, hkv, d, dtype=dtype, kv_dtype=kv, seed=hq + d + len(news))
    out = torch.full_like(c["q"], float("nan"))
    names = kernels_of(lambda: ops.append_prefill_attn(
        out, c["q"], None, None, c["k_pool"], c["v_pool"], None, c["table"], c["ctx"], c["cu"], c["scale"], max(news), c["ks"],
        c["vs"], None, lens(len(news), longest)))
    assert any(kernel in n for n in names), names
    if kernel == ROWS:
        groups, tiles = hq // (hq // hkv), sum(-(-n * (hq // hkv) // 128) for n in news)
        assert any(f", {4 if groups * tiles > 32 and d == 128 else 8}>" in n for n in names if ROWS in n), names
    assert_close_attn(to_f64(out), tp.oracle(c), 1e-2, 2e-2, f"{hq}/{hkv} {d} {priors} {news}")


def test_unknown_contexts_count_as_the_table(device):
    """Without host lengths the table's width stands for them, and a plan's steps hand theirs along."""
    import aicomp_amd.block_manager as bm
    c = tp.build_case(device, [0], [24], 8, 8, 128, seed=1)
    wide = torch.zeros(1, 64, dtype=torch.int32, device=device)
    wide[:, :c["table"].shape[1]] = c["table"]
    out = torch.empty_like(c["q"])

    def step(table, host_lens=None):
        ops.append_prefill_attn(out, c["q"], None, None, c["k_pool"], c["v_pool"], None, table, c["ctx"], c["cu"], c["scale"], 24,
                                None, None, None, host_lens)

    assert any(TILES in n for n in kernels_of(lambda: step(c["table"])))
    assert any(ROWS in n for n in kernels_of(lambda: step(wide)))
    assert any(TILES in n for n in kernels_of(lambda: step(wide, np.asarray([24], dtype=np.int32))))
    planner = bm.StepPlanner(80, 16, max_seqs=2, max_seq_len=1024, prefill_chunk=24, device=device)
    planner.add_request("a", 300)
    pools = [torch.zeros(80, 8, 16, 128, dtype=torch.bfloat16, device=device) for _ in range(2)]
    for i in range(12):
        plan = planner.schedule()
        names = kernels_of(lambda: bm.paged_attention_step(plan, out, c["q"], c["q"], c["q"], *pools, 0.1))
        assert any((TILES if 24 * (i + 1) < 256 else ROWS) in n for n in names), (i, names)
