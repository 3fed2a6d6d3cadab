"""A layer's decode step in one launch (rotary embedding, append, attention) against the two calls it stands for: the
same bits in the output and in the pools."""
import math

import numpy as np
import pytest
import torch

from aicomp_amd import _lib, ops
from helpers import kernels_of

pytestmark = [pytest.mark.gpu, pytest.mark.routing("library")]
CTX = [1, 2, 16, 17, 31, 32, 33, 63, 64, 65, 128, 129, 300, 7]


def _case(device, dtype, kv, hq, hkv, d, ctx, seed):
    g = torch.Generator().manual_seed(seed)
    B, need = len(ctx), [-(-n // 16) for n in ctx]
    nb = sum(need) + 3
    table, perm, at = torch.zeros(B, max(need) + 2, dtype=torch.int32), torch.randperm(nb, generator=g), 0
    for s, n in enumerate(need):
        table[s, :n] = perm[at:at + n].to(torch.int32)
        at += n
    pools, scales = [], [None, None]
    for i in range(2):
        x = torch.randn(nb, hkv, 16, d, generator=g) * 0.5
        if kv == torch.float8_e4m3fn:
            scales[i] = torch.full((hkv,), 2.75 / 448).to(device)
            x = (x / (2.75 / 448)).clamp(-448, 448)
        pools.append(x.to(kv).to(device))
    qkv = (torch.randn(B, hq + 2 * hkv, d, generator=g) * 0.7).to(dtype).to(device)
    cos, sin = ops.rotary_tables(1.0 / 10000 ** (torch.arange(0, d, 2) / d).to(device), 512, dtype)
    lens = np.asarray(ctx, dtype=np.int32)
    slots = torch.tensor([int(table[s, (n - 1) // 16]) * 16 + (n - 1) % 16 for s, n in enumerate(ctx)])
    return dict(q=qkv[:, :hq], k=qkv[:, hq:hq + hkv], v=qkv[:, hq + hkv:], cos=cos, sin=sin,
                pos=torch.tensor([n - 1 for n in ctx]).to(device), slots=slots.to(device), table=table.to(device),
                ctx=torch.from_numpy(lens).to(device), lens=lens, pools=pools, scales=scales, scale=1 / math.sqrt(d))


def _bits(t):
    return t.view({1: torch.uint8, 2: torch.int16, 4: torch.int32}[t.element_size()])


def _one(c, lens):
    kp, vp = (p.clone() for p in c["pools"])
    out = ops.rope_paged_decode_attn(c["q"], c["k"], c["v"], c["cos"], c["sin"], c["pos"], kp, vp, c["slots"], c["table"],
                                     c["ctx"], lens, c["scale"], *c["scales"])
    return out, kp, vp


def _two(c, width):
    kp, vp = (p.clone() for p in c["pools"])
    q, out = torch.empty_like(c["q"].contiguous()), torch.empty_like(c["q"].contiguous())
    ops.rope_kv_append(c["q"], c["k"], c["v"], c["cos"], c["sin"], c["pos"], kp, vp, c["slots"], *c["scales"], query_out=q)
    ops.paged_decode_attn(out, q, kp, vp, c["table"][:, :width], c["ctx"], c["scale"], *c["scales"])
    return out, kp, vp


KINDS = [(torch.bfloat16, None), (torch.float16, None), (torch.float32, None), (torch.bfloat16, torch.float8_e4m3fn),
         (torch.float16, torch.float8_e4m3fn)]


@pytest.mark.parametrize("dtype,kv", KINDS)
@pytest.mark.parametrize("hq,hkv,d", [(4, 4, 64), (8, 2, 64), (16, 2, 64), (8, 2, 128), (10, 2, 128), (32, 2, 128)])
def test_one_launch_equals_two(device, decode_routing, dtype, kv, hq, hkv, d):
    c = _case(device, dtype, kv or dtype, hq, hkv, d, CTX, hq + d)
    for lens, width in ((c["lens"], 19), (None, c["table"].shape[1])):
        for got, want in zip(_one(c, lens), _two(c, width)):
            assert torch.equal(_bits(got), _bits(want)), (width,)


@pytest.mark.parametrize("dtype,kv,hq,hkv,d,longest", [
    (torch.bfloat16, None, 8, 2, 128, 600), (torch.float16, None, 4, 4, 128, 513), (torch.bfloat16, torch.float8_e4m3fn, 8, 2, 128, 600),
    (torch.float16, torch.float8_e4m3fn, 16, 2, 128, 640), (torch.bfloat16, None, 8, 2, 64, 1100), (torch.float16, None, 16, 2, 64, 1280),
    (torch.float32, None, 8, 2, 64, 640), (torch.float32, None, 16, 2, 64, 600), (torch.float32, None, 8, 2, 128, 400),
    (torch.float32, None, 16, 2, 128, 448)])
def test_rows_of_eight_waves(device, decode_routing, dtype, kv, hq, hkv, d, longest):
    """Rows that are whole and long in few workgroups."""
    c = _case(device, dtype, kv or dtype, hq, hkv, d, [longest, 1, longest - 17, 65, 255, 256, 257], hq + d)
    c["cos"], c["sin"] = ops.rotary_tables(1.0 / 10000 ** (torch.arange(0, d, 2) / d).to(device), 1300, dtype)
    got = []
    names = [n for n in kernels_of(lambda: got.extend(_one(c, c["lens"]))) if "paged_decode" in n]
    assert len(names) == 1 and "8, true>" in names[0], names
    for a, b in zip(got, _two(c, -(-longest // 16))):
        assert torch.equal(_bits(a), _bits(b))


@pytest.mark.parametrize("dtype,kv,d", [(torch.bfloat16, None, 64), (torch.float32, None, 128), (torch.float16, torch.float8_e4m3fn, 128)])
def test_split_rows_and_odd_slots(device, decode_routing, dtype, kv, d):
    """Rows of several partitions; a padding row, a row stored elsewhere, one without a table row, an empty one."""
    c = _case(device, dtype, kv or dtype, 8, 2, d, [1500, 1, 800, 257, 40, 33], 3)
    c["cos"], c["sin"] = ops.rotary_tables(1.0 / 10000 ** (torch.arange(0, d, 2) / d).to(device), 1600, dtype)
    for got, want in zip(_one(c, c["lens"]), _two(c, 94)):
        assert torch.equal(_bits(got), _bits(want))
    used = set(c["table"][:, :94].flatten().tolist())
    spare = next(b for b in range(c["pools"][0].shape[0]) if b not in used)
    c["slots"][1], c["slots"][2], c["pos"][3] = -1, spare * 16 + 5, 5000
    c["ctx"][4] = 0
    got, want = _one(c, c["lens"]), _two(c, 94)
    rows = [0, 1, 2, 4, 5]
    assert torch.equal(_bits(got[0][rows]), _bits(want[0][rows]))
    assert torch.equal(_bits(got[1]), _bits(want[1])) and torch.equal(_bits(got[2]), _bits(want[2]))


def test_what_it_declines(device, decode_routing):
    """Batches for the balanced schedule, many split rows, other head dims, rows that cannot be read in vectors: None, and nothing written."""
    c = _case(device, torch.bfloat16, torch.bfloat16, 8, 2, 64, CTX, 1)
    prev = ops.set_small_decode_tokens(0)
    try:
        assert _one(c, c["lens"])[0] is None
    finally:
        ops.set_small_decode_tokens(prev)
    odd = torch.empty(c["q"].numel() + 1, dtype=torch.bfloat16, device=device)[1:].view(c["q"].shape)
    odd.copy_(c["q"])
    c["q"] = odd
    out, kp, vp = _one(c, c["lens"])
    assert out is None and torch.equal(_bits(kp), _bits(c["pools"][0])) and torch.equal(_bits(vp), _bits(c["pools"][1]))
    # split rows of more than 512 workgroups, but for float32 groups of up to four heads
    for dtype, kv, hq, rows, one in ((torch.bfloat16, torch.float8_e4m3fn, 8, 21, True), (torch.bfloat16, torch.float8_e4m3fn, 8, 22, False),
                                     (torch.float32, torch.float32, 32, 22, True), (torch.float32, torch.float32, 40, 22, False)):
        s = _case(device, dtype, kv, hq, 8, 64, [641] * rows, 3)
        s["cos"], s["sin"] = ops.rotary_tables(1.0 / 10000 ** (torch.arange(0, 64, 2) / 64).to(device), 700, dtype)
        got = _one(s, s["lens"])
        assert (got[0] is not None) == one
        if one:
            for a, b in zip(got, _two(s, 41)):
                assert torch.equal(_bits(a), _bits(b))
    w = _case(device, torch.bfloat16, torch.bfloat16, 4, 2, 256, [5, 20], 2)
    assert _one(w, w["lens"])[0] is None
    w["table"] = w["table"].long()
    assert _one(w, w["lens"])[0] is None
    lib = _lib.load()
    assert lib.aicomp_rope_paged_decode_attn(*([None] * 2), 0, 0, None, None, 0, 0, None, None, 0, 0, *([None] * 5), 0, None, 1,
                                             4, 2, 64, 16, 1, 4, 1.0, 1, 1, None, None, None, 0, None) == 1


@pytest.mark.parametrize("dtype,kv,d", [(torch.bfloat16, None, 64), (torch.float32, None, 128), (torch.float16, torch.float8_e4m3fn, 128)])
@pytest.mark.parametrize("known", [1, 40, 300, 900, 1500])
def test_lengths_on_the_host_only_size_the_call(device, decode_routing, dtype, kv, d, known):
    """Rows that have grown past what the host knows of them: in full, whether the call is sized for whole rows (1 to 300
    tokens) or for partitions; against a call that is sized for the table."""
    c = _case(device, dtype, kv or dtype, 8, 2, d, [1500, 1, 800, 257, 40, 33], 4)
    c["cos"], c["sin"] = ops.rotary_tables(1.0 / 10000 ** (torch.arange(0, d, 2) / d).to(device), 1600, dtype)
    got, want = _one(c, np.minimum(c["lens"], known)), _two(c, c["table"].shape[1])
    # float32 sums and weights in another order, then the output's own rounding
    tol = 2e-6 if dtype == torch.float32 else 2e-3
    assert (got[0].float() - want[0].float()).abs().max().item() <= tol
    assert torch.equal(_bits(got[1]), _bits(want[1])) and torch.equal(_bits(got[2]), _bits(want[2]))


@pytest.mark.parametrize("dtype,kv", KINDS)
def test_a_slot_that_is_read_takes_two_calls(device, decode_routing, dtype, kv):
    """Rows whose slot is an earlier place of their own sequence, or the last one of another's: the append comes first, as in
    the two calls; a padding row does not stand in the way of the one launch."""
    import aicomp_amd.block_manager as bm
    from aicomp_amd.generation import PagedAttentionBackend
    c = _case(device, dtype, kv or dtype, 8, 2, 64, [70, 33, 18, 129], 5)
    B, host_table, slots = 4, c["table"].cpu().numpy(), c["slots"].cpu().numpy()
    backend = PagedAttentionBackend(1, c["pools"][0].shape[0], 2, 64, dtype=dtype, device=device, kv_dtype=kv,
                                    inv_freq=1.0 / 10000 ** (torch.arange(0, 64, 2) / 64).to(device), max_positions=512)
    if kv is not None:
        backend.set_scales(0, *c["scales"])
    for slot, one in ((None, True), (-1, True), (host_table[0, 1] * 16 + 3, False), (slots[3], False)):
        s = slots.copy()
        if slot is not None:
            s[0] = slot
        if slot == slots[3]:
            s[3] = -1
        c["slots"] = torch.from_numpy(s).to(device)
        backend.k_pools[0], backend.v_pools[0] = (p.clone() for p in c["pools"])
        assert one == (ops.rope_paged_decode_attn(
            c["q"], c["k"], c["v"], c["cos"], c["sin"], c["pos"], c["pools"][0].clone(), c["pools"][1].clone(), c["slots"],
            c["table"], c["ctx"], c["lens"], c["scale"], *c["scales"], s, host_table) is not None)
        cu = np.arange(B + 1, dtype=np.int32)
        backend.begin_step(bm.StepPlan(
            seq_ids=list(range(B)), num_prefill_seqs=0, new_lens=np.ones(B, dtype=np.int32), max_q_len=0, total_new_tokens=B,
            block_table=c["table"], context_lens=c["ctx"], cu_q_lens=torch.from_numpy(cu).to(device), slot_mapping=c["slots"],
            positions=c["pos"], preempted=[], host_block_table=host_table, host_context_lens=c["lens"], host_cu_q_lens=cu,
            host_slot_mapping=s, host_positions=c["lens"].astype(np.int64) - 1))
        out = backend.attend(0, c["q"], c["k"], c["v"])
        want = _two(c, c["table"].shape[1] if not one else 9)
        assert torch.equal(_bits(out), _bits(want[0])), slot
        assert torch.equal(_bits(backend.k_pools[0]), _bits(want[1])) and torch.equal(_bits(backend.v_pools[0]), _bits(want[2]))


@pytest.mark.parametrize("dtype,kv,d", [(torch.bfloat16, None, 64), (torch.float32, None, 128), (torch.float16, torch.float8_e4m3fn, 128)])
def test_a_recorded_launch_is_sized_for_the_table(device, decode_routing, dtype, kv, d):
    """Recorded while the rows are short, replayed as they grow: the bits of the two calls over the whole table each time."""
    c = _case(device, dtype, kv or dtype, 8, 2, d, [1500, 40, 800, 257], 6)
    c["cos"], c["sin"] = ops.rotary_tables(1.0 / 10000 ** (torch.arange(0, d, 2) / d).to(device), 1600, dtype)
    full, table = c["lens"].copy(), c["table"].cpu().numpy()

    def at(lens):                                            # the rows as they are at these lengths
        c["ctx"].copy_(torch.from_numpy(lens))
        c["pos"].copy_(torch.from_numpy(lens.astype(np.int64) - 1))
        c["slots"].copy_(torch.from_numpy(table[range(4), (lens - 1) // 16].astype(np.int64) * 16 + (lens - 1) % 16))

    short = np.minimum(full, [30, 20, 10, 33]).astype(np.int32)
    at(short)
    _one(c, short)
    kp, vp = (p.clone() for p in c["pools"])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.rope_paged_decode_attn(c["q"], c["k"], c["v"], c["cos"], c["sin"], c["pos"], kp, vp, c["slots"], c["table"],
                                         c["ctx"], short, c["scale"], *c["scales"])
    for lens in (short, np.minimum(full, 300), np.minimum(full, 1000), full):
        at(lens)
        for pool, first in zip((kp, vp), c["pools"]):
            pool.copy_(first)
        graph.replay()
        torch.cuda.synchronize()
        for got, want in zip((out, kp, vp), _two(c, c["table"].shape[1])):
            assert torch.equal(_bits(got), _bits(want)), lens
