"""aicomp_paged_decode_attn_append_static: the decode step for callers that cannot allocate.

Called through the C ABI (ctypes, raw device pointers) and compared bit for bit, output and
pools, with aicomp_paged_decode_attn_append on a workspace of the caller's: two calls in a row
on the same GPU, the second with a smaller batch and shorter contexts, so that the second call
runs over whatever the first left in the library's scratch array.
"""
import math

import pytest
import torch

from aicomp_amd import _lib

pytestmark = pytest.mark.gpu

STATIC_SCRATCH_BYTES = 32 << 20


def _case(device, seed, B, hq, hkv, d, ctx_lo, ctx_hi, kv_dtype):
    g = torch.Generator().manual_seed(seed)
    ctx = torch.randint(ctx_lo, ctx_hi + 1, (B,), generator=g)          # lengths including the new token
    width = math.ceil(ctx_hi / 16) + 1
    nb = B * width + 5
    table = torch.randperm(nb, generator=g)[: B * width].reshape(B, width).to(torch.int32)
    k = torch.randn(nb, hkv, 16, d, generator=g) * 0.5
    v = torch.randn(nb, hkv, 16, d, generator=g) * 0.5
    ks = vs = None
    if kv_dtype == torch.float8_e4m3fn:
        ks = torch.full((hkv,), 2.5 / 448, dtype=torch.float32, device=device)
        vs = torch.full((hkv,), 2.5 / 448, dtype=torch.float32, device=device)
        k, v = (k / (2.5 / 448)).clamp(-448, 448), (v / (2.5 / 448)).clamp(-448, 448)
    return dict(B=B, hq=hq, hkv=hkv, d=d, nb=nb, width=width, kv_dtype=kv_dtype,
                table=table.to(device), ctx=ctx.to(torch.int32).to(device),
                k=k.to(kv_dtype).to(device), v=v.to(kv_dtype).to(device), ks=ks, vs=vs,
                q=torch.randn(B, hq, d, generator=g).to(torch.bfloat16).to(device),
                nk=(torch.randn(B, hkv, d, generator=g) * 0.5).to(torch.bfloat16).to(device),
                nv=(torch.randn(B, hkv, d, generator=g) * 0.5).to(torch.bfloat16).to(device))


def _ptr(t):
    return None if t is None else t.data_ptr()


def _run(lib, c, partition_size, static):
    """One fused append + decode call on copies of the case's pools; returns (out, k_pool, v_pool)."""
    k, v = c["k"].clone(), c["v"].clone()
    out = torch.full_like(c["q"], float("nan"))
    kd = _lib.FP8_E4M3 if c["kv_dtype"] == torch.float8_e4m3fn else _lib.BF16
    stream = torch.cuda.current_stream().cuda_stream
    head = (out.data_ptr(), c["q"].data_ptr(), c["nk"].data_ptr(), c["nv"].data_ptr(), c["nk"].stride(0),
            c["nk"].stride(1), k.data_ptr(), v.data_ptr(), c["table"].data_ptr(), c["table"].stride(0),
            c["ctx"].data_ptr(), c["B"], c["hq"], c["hkv"], c["d"], 16, c["width"], c["nb"],
            1.0 / math.sqrt(c["d"]), _lib.BF16, kd, _ptr(c["ks"]), _ptr(c["vs"]), partition_size)
    if static:
        rc = lib.aicomp_paged_decode_attn_append_static(*head, stream)
    else:
        need = lib.aicomp_paged_decode_workspace_bytes(c["B"], c["hq"], c["hkv"], c["d"], 16, c["width"],
                                                       _lib.BF16, kd, partition_size)
        ws = torch.empty(max(need, 16), dtype=torch.uint8, device=out.device)
        rc = lib.aicomp_paged_decode_attn_append(*head, ws.data_ptr(), need, stream)
    _lib.check(rc, lib)
    torch.cuda.synchronize()
    return out, k, v


def _same(a, b):
    return torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("kv_dtype,d,partition_size", [
    (torch.bfloat16, 128, 0),             # balanced schedule: partials and row records in the scratch
    (torch.float8_e4m3fn, 128, 0),
    (torch.bfloat16, 128, 256),           # grid schedule, explicit split
    (torch.bfloat16, 64, 0),              # head_dim 64
])
def test_static_scratch_call_equals_workspace_call_twice_in_a_row(device, kv_dtype, d, partition_size):
    lib = _lib.load()
    big = _case(device, 11, B=24, hq=32, hkv=8, d=d, ctx_lo=300, ctx_hi=2500, kv_dtype=kv_dtype)
    small = _case(device, 12, B=5, hq=32, hkv=8, d=d, ctx_lo=1, ctx_hi=700, kv_dtype=kv_dtype)
    for name, c in (("first call", big), ("second, smaller call", small)):
        print(f"static-scratch decode: {name}, B={c['B']} d={d} kv={kv_dtype} partition={partition_size}", flush=True)
        got = _run(lib, c, partition_size, static=True)
        want = _run(lib, c, partition_size, static=False)
        assert not torch.isnan(got[0].float()).any(), f"{name}: output rows left unwritten"
        assert _same(got[0], want[0]), f"{name}: output differs from the workspace call"
        assert _same(got[1], want[1]) and _same(got[2], want[2]), f"{name}: pools differ from the workspace call"
        # the new rows did reach the pools
        assert not _same(got[1], c["k"]), f"{name}: K pool unchanged"


def test_static_scratch_refuses_shapes_beyond_its_size(device):
    lib = _lib.load()
    # 1024 sequences at 64 / 8 heads need far more than 32 MiB of partials
    need = lib.aicomp_paged_decode_workspace_bytes(1024, 64, 8, 128, 16, 64, _lib.BF16, _lib.BF16, 0)
    assert need > STATIC_SCRATCH_BYTES
    x = torch.zeros(16, dtype=torch.int32, device=device)        # never dereferenced: the size check comes first
    p = x.data_ptr()
    rc = lib.aicomp_paged_decode_attn_append_static(p, p, p, p, 1024, 128, p, p, p, 64, p, 1024, 64, 8, 128, 16,
                                                    64, 4096, 0.1, _lib.BF16, _lib.BF16, None, None, 0, None)
    assert rc == 4 and b"built-in scratch" in lib.aicomp_kv_last_error()


@pytest.mark.routing("balanced")
@pytest.mark.parametrize("B,hq,hkv,longest", [(32, 16, 1, 2048), (1024, 64, 4, 64)])
def test_static_scratch_takes_float32_batches_whose_balanced_partials_do_not_fit(device, B, hq, hkv, longest):
    """The balanced schedule's partials (34 and 66 MiB here) are more than the array holds, the grid schedule's
    (8 MiB, none) are not: the call is accepted, and is the grid schedule's, bit for bit."""
    import test_gpu_prefill as tp
    lib, d, F32 = _lib.load(), 128, _lib.F32
    ctx = [1 + (i * 977) % longest for i in range(B - 1)] + [longest]
    c = tp.build_case(device, [n - 1 for n in ctx], [1] * B, hq, hkv, d, dtype=torch.float32, seed=B, poison="all")
    rows = torch.arange(B, device=device)
    blk, at = c["table"][rows, (c["ctx"] - 1).long() // 16].long(), (c["ctx"] - 1).long() % 16
    nk, nv = c["k_pool"][blk, :, at].clone(), c["v_pool"][blk, :, at].clone()
    width = c["table"].shape[1]
    assert lib.aicomp_paged_decode_workspace_bytes(B, hq, hkv, d, 16, width, F32, F32, 0) > STATIC_SCRATCH_BYTES
    outs = []
    for static in (True, False):
        kp, vp = c["k_pool"].clone(), c["v_pool"].clone()
        kp[blk, :, at], vp[blk, :, at] = float("nan"), float("nan")
        out = torch.full_like(c["q"], float("nan"))
        head = (out.data_ptr(), c["q"].data_ptr(), nk.data_ptr(), nv.data_ptr(), nk.stride(0), nk.stride(1), kp.data_ptr(),
                vp.data_ptr(), c["table"].data_ptr(), c["table"].stride(0), c["ctx"].data_ptr(), B, hq, hkv, d, 16, width,
                kp.shape[0], c["scale"], F32, F32, None, None)
        stream = torch.cuda.current_stream().cuda_stream
        if static:
            rc = lib.aicomp_paged_decode_attn_append_static(*head, 0, stream)
        else:
            ps = 64 if longest == 2048 else 1024
            ws = torch.empty(max(16, lib.aicomp_paged_decode_workspace_bytes(B, hq, hkv, d, 16, width, F32, F32, ps)),
                             dtype=torch.uint8, device=device)
            rc = lib.aicomp_paged_decode_attn_append(*head, ps, ws.data_ptr(), ws.numel(), stream)
        _lib.check(rc, lib)
        torch.cuda.synchronize()
        outs.append((out, kp, vp))
    (a, ka, va), (b, kb, vb) = outs
    assert torch.isfinite(a).all() and _same(a, b) and _same(ka, kb) and _same(va, vb)
    assert _same(ka, c["k_pool"]) and _same(va, c["v_pool"])                # the new rows are where they were taken from
    # plain attention of every sixteenth row in float64; 1e-5: the bound of test_gpu_decode_f32
    for r in range(0, B, 16):
        n = ctx[r]
        ids = c["table"][r, :-(-n // 16)].long()
        k, v = (p[ids].transpose(1, 2).reshape(-1, hkv, d)[:n].double() for p in (c["k_pool"], c["v_pool"]))
        q = c["q"][r].double().view(hkv, hq // hkv, d)
        w = torch.softmax((q[:, :, None] * k.transpose(0, 1)[:, None]).sum(-1) * c["scale"], -1)
        want = (w[..., None] * v.transpose(0, 1)[:, None]).sum(2).view(hq, d)
        assert (a[r].double() - want).abs().max().item() <= 1e-5
