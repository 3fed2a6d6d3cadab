"""Rotary + append at the edges of the launch shapes: head counts that do not fill a workgroup's passes or
need several slices, the token count where a lane takes two heads, head dims of both kernels, against the
oracle bit for bit."""
import pytest
import torch

from aicomp_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,d", [(1, 1, 64), (3, 1, 128), (16, 2, 128), (5, 5, 64), (32, 8, 128), (64, 8, 128), (7, 1, 96)])
@pytest.mark.parametrize("T", [1, 255, 256])
@pytest.mark.parametrize("kv", [None, torch.float8_e4m3fn])
def test_launch_shapes(device, hq, hkv, d, T, kv):
    _check(device, hq, hkv, d, T, torch.bfloat16, kv)


# More KV heads than one pass of a workgroup holds (16 of D 128, 32 of D 64): both heads of a lane are V heads, or both K
@pytest.mark.parametrize("hq,hkv,d", [(32, 32, 128), (20, 20, 128), (40, 40, 64), (17, 17, 128)])
@pytest.mark.parametrize("T", [255, 256, 300])
@pytest.mark.parametrize("dtype,kv", [(torch.bfloat16, None), (torch.float16, None), (torch.float32, None),
                                      (torch.bfloat16, torch.float8_e4m3fn)])
def test_more_kv_heads_than_a_pass(device, hq, hkv, d, T, dtype, kv):
    _check(device, hq, hkv, d, T, dtype, kv)


def _check(device, hq, hkv, d, T, dtype, kv):
    g = torch.Generator().manual_seed(hq + d + T)
    qkv = torch.randn(T, hq + 2 * hkv, d, generator=g).to(dtype).to(device)
    q, k, v = qkv[:, :hq], qkv[:, hq:hq + hkv], qkv[:, hq + hkv:]
    cos, sin = ops.rotary_tables(1.0 / 10000.0 ** (torch.arange(0, d, 2) / d), 512, dtype, device=device)
    pos = torch.randint(0, 512, (T,), generator=g).to(device)
    blocks = T // 16 + 3
    slots = torch.randperm(blocks * 16, generator=g)[:T]
    slots[T // 2] = -1                                             # a padding row: Q is rotated, nothing is stored
    slots = slots.to(device)
    ks = vs = None
    if kv is not None:
        ks, vs = (torch.rand(hkv, generator=g).to(device) * 0.01 + 0.005 for _ in range(2))
    kp, vp = (torch.zeros(blocks, hkv, 16, d, dtype=kv or dtype, device=device) for _ in range(2))
    out = torch.empty(T, hq, d, dtype=dtype, device=device)
    ops.rope_kv_append(q, k, v, cos, sin, pos, kp, vp, slots, ks, vs, query_out=out)
    # torch's own evaluation of the same expression, one rounding per product and sum
    half = lambda x: torch.cat((-x[..., d // 2:], x[..., :d // 2]), -1)
    rot = lambda x: x * cos[pos][:, None] + half(x) * sin[pos][:, None]
    kp2, vp2 = torch.zeros_like(kp), torch.zeros_like(vp)
    ops.kv_append(rot(k).contiguous(), v.contiguous(), kp2, vp2, slots, ks, vs)
    bits = lambda t: t.view({1: torch.uint8, 2: torch.int16, 4: torch.int32}[t.element_size()])
    assert torch.equal(bits(out), bits(rot(q)))
    assert torch.equal(bits(kp), bits(kp2)) and torch.equal(bits(vp), bits(vp2))


def test_more_tokens_than_a_launch_of_one_per_workgroup_holds(device):
    """2^26 + 3 tokens of one head: rounded up to whole waves they are more than the 2^32 lanes of a launch
    dimension.  The same row for every token (stride 0); the first, a middle and the last one are stored."""
    T, d, dtype = (1 << 26) + 3, 64, torch.bfloat16
    g = torch.Generator().manual_seed(1)
    row = torch.randn(3, 1, 1, d, generator=g).to(dtype).to(device)
    q, k, v = (row[i].expand(T, 1, d) for i in range(3))
    cos, sin = ops.rotary_tables(1.0 / 10000.0 ** (torch.arange(0, d, 2) / d), 8, dtype, device=device)
    slots = torch.full((T,), -1, dtype=torch.int64, device=device)
    at = [0, (1 << 26) - 1, T - 1]
    slots[at] = torch.tensor([3, 17, 30], device=device)
    kp, vp = (torch.zeros(2, 1, 16, d, dtype=dtype, device=device) for _ in range(2))
    out = torch.zeros(1, 1, d, dtype=dtype, device=device)
    ops.rope_kv_append(q, k, v, cos, sin, torch.full((T,), 5, device=device), kp, vp, slots, query_out=out.expand(T, 1, d))
    kp2, vp2, out2 = torch.zeros_like(kp), torch.zeros_like(vp), torch.empty(3, 1, d, dtype=dtype, device=device)
    ops.rope_kv_append(q[:3], k[:3], v[:3], cos, sin, torch.full((3,), 5, device=device), kp2, vp2, slots[at], query_out=out2)
    assert torch.equal(out, out2[:1]) and torch.equal(kp, kp2) and torch.equal(vp, vp2) and bool(kp.any())
