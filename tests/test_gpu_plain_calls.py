"""The plain calls of ``aicomp_amd.ops`` by their native host route and by the ctypes one: the same
results, and the same refusals."""
import pytest
import torch

from aicomp_amd import ops

BF, F8 = torch.bfloat16, torch.float8_e4m3fn


def _inputs(dev, kv=BF, hq=8, hkv=2, d=64, lens=(5, 40, 17)):
    torch.manual_seed(3)
    S, T, blocks = len(lens), sum(lens), 16
    mk = lambda *s: torch.randn(*s, device=dev).to(BF)
    table = torch.randperm(blocks, device=dev)[:S * 4].view(S, 4).to(torch.int32)
    pos = torch.cat([torch.arange(n, device=dev) for n in lens])
    seq = torch.cat([torch.full((n,), s, device=dev) for s, n in enumerate(lens)])
    slots = table[seq, pos // 16].long() * 16 + pos % 16
    qkv = mk(T, hq + 2 * hkv, d)
    pools = [torch.zeros(blocks, hkv, 16, d, device=dev, dtype=torch.uint8 if kv == F8 else kv) for _ in range(2)]
    pools = [p.view(F8) if kv == F8 else p for p in pools]
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device=dev)
    cos, sin = ops.rotary_tables(torch.rand(d // 2, device=dev), 64, BF)
    scales = [torch.full((hkv,), 0.02, device=dev) for _ in range(2)] if kv == F8 else [None, None]
    return dict(q=qkv[:, :hq], k=qkv[:, hq:hq + hkv], v=qkv[:, hq + hkv:], kp=pools[0], vp=pools[1], table=table, slots=slots,
                pos=pos, cu=cu, ctx=torch.tensor(lens, dtype=torch.int32, device=dev), cos=cos, sin=sin, ks=scales[0],
                vs=scales[1], longest=max(lens), logits=mk(3, 1000).float(), u=torch.rand(3, device=dev))


def _everything(a):
    q = torch.empty(a["q"].shape, dtype=BF, device=a["q"].device)
    ops.kv_append(a["k"], a["v"], a["kp"], a["vp"], a["slots"], a["ks"], a["vs"])
    first = a["kp"].clone()
    ops.rope_kv_append(a["q"], a["k"], a["v"], a["cos"], a["sin"], a["pos"], a["kp"], a["vp"], a["slots"], a["ks"], a["vs"],
                       query_out=q)
    pre = ops.paged_prefill_attn(torch.empty_like(q), q, a["kp"], a["vp"], a["table"], a["ctx"], a["cu"], 0.125,
                                 a["longest"], a["ks"], a["vs"])
    rows, new = q[:3].contiguous(), (a["k"][:3], a["v"][:3])
    dec = ops.paged_decode_attn(torch.empty_like(rows), rows, a["kp"], a["vp"], a["table"], a["ctx"], 0.125, a["ks"], a["vs"])
    fused = ops.paged_decode_attn(torch.empty_like(rows), rows, a["kp"], a["vp"], a["table"], a["ctx"], 0.125, a["ks"],
                                  a["vs"], partition_size=16, new_key=new[0], new_value=new[1])
    tokens = ops.sample_tokens(a["logits"], 0.8, 20, 0.9, uniforms=a["u"])
    greedy = ops.sample_tokens(a["logits"], do_sample=False)
    return [t.view(torch.uint8) if t.dtype == F8 else t for t in (first, q, pre, dec, fused, a["kp"], a["vp"], tokens, greedy)]


@pytest.mark.gpu
@pytest.mark.parametrize("kv", [BF, F8])
def test_native_and_ctypes_routes_agree(device, monkeypatch, kv):
    assert ops._FAST is not None, "aicomp_amd/_aicomp_fast is not built"
    native = _everything(_inputs(device, kv))
    monkeypatch.setattr(ops, "_FAST", None)
    for a, b in zip(native, _everything(_inputs(device, kv))):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("change", [
    dict(slots=lambda t: t.int()), dict(slots=lambda t: t[:-1]), dict(k=lambda t: t.float()), dict(k=lambda t: t[:, :1]),
    dict(kp=lambda t: t.transpose(0, 1)), dict(ctx=lambda t: t.long()), dict(table=lambda t: t[:2]), dict(cu=lambda t: t[:-1]),
    dict(pos=lambda t: t.cpu()), dict(cos=lambda t: t.float()), dict(u=lambda t: t[:2]), dict(vp=lambda t: t.half()),
    dict(logits=lambda t: t.t()),
], ids=lambda c: next(iter(c)))
def test_refusals_are_the_same_by_both_routes(device, monkeypatch, change):
    said = []
    for native in (True, False):
        a = _inputs(device)
        for name, f in change.items():
            a[name] = f(a[name])
        with monkeypatch.context() as m:
            if not native:
                m.setattr(ops, "_FAST", None)
            with pytest.raises(RuntimeError) as e:
                _everything(a)
        said.append(str(e.value))
    assert said[0] == said[1]


@pytest.mark.gpu
def test_strided_rows_are_still_converted(device):
    """Rows whose last dimension is not contiguous are copied, as they always were."""
    a = _inputs(device)
    k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (a["k"], a["v"]))
    assert k.stride(2) != 1
    ops.kv_append(k, v, a["kp"], a["vp"], a["slots"])
    want = _inputs(device)
    ops.kv_append(want["k"], want["v"], want["kp"], want["vp"], want["slots"])
    assert torch.equal(a["kp"], want["kp"]) and torch.equal(a["vp"], want["vp"])


@pytest.mark.gpu
def test_two_threads_on_one_stream_share_the_scratch(device):
    """Calls of two launches (decode and merge) from two host threads on one stream, one through the operator's
    lean route and one through the plain call: each gets what it gets alone, bit for bit, every time."""
    import threading

    from aicomp_amd import kv_cache as akv
    from aicomp_amd import _aicomp_fast as fast
    torch.manual_seed(5)
    B, hq, hkv, d, n, rounds = 4, 8, 2, 64, 2000, 400
    layer = akv._PagedLayer(B, hkv, d, 2048, BF, device)
    layer.append(*(torch.randn(B, hkv, n, d, device=device).to(BF) for _ in range(2)), 0, 1)
    handle = fast.layer(layer.k_pool, layer.v_pool, layer.block_table, layer.ctx_rows)
    q = torch.randn(B, hq, 1, d, device=device).to(BF)
    new = [torch.randn(B, hkv, 1, d, device=device).to(BF) for _ in range(2)]
    other = [t.clone() for t in (layer.k_pool, layer.v_pool)]
    rows, lens = torch.randn(B, hq, d, device=device).to(BF), torch.tensor([1999, 700, 1300, 1], dtype=torch.int32, device=device)
    calls = [lambda: fast.decode_step(handle, q, *new, n, 1, 0.125).view(B, hq, d),
             lambda: ops.paged_decode_attn(torch.empty_like(rows), rows, *other, layer.block_table, lens, 0.125)]
    assert all(ops.decode_workspace_bytes(B, hq, hkv, d, 16, w, BF, BF) > 0 for w in (126, 128))
    want = [f() for f in calls]
    torch.cuda.synchronize()
    got, go = [[], []], threading.Barrier(2)

    def run(i):
        go.wait()
        got[i] += [calls[i]() for _ in range(rounds)]

    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i in range(2):
        assert len(got[i]) == rounds and all(torch.equal(x, want[i]) for x in got[i])
