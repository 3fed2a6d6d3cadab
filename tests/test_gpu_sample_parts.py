"""Rows cut into parts against the one-launch kernel: the same tokens and kept sets.  The one-launch
kernel's walk over a whole row (a row with fewer finite logits than k) rounds 1 / mass to float32 before the
product, its candidate list does not: two roundings of 2^-24 apart at most."""
import pytest
import torch

from aicomp_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _one_launch(x, temperature, top_k, top_p, do_sample, u):
    lib = _lib.load()
    out = torch.empty(x.shape[0], dtype=torch.int64, device=x.device)
    probs = torch.empty(x.shape, dtype=torch.float32, device=x.device)
    rc = lib.aicomp_sample_tokens(out.data_ptr(), x.data_ptr(), x.stride(0), probs.data_ptr(), u.data_ptr(), *x.shape,
                                  temperature, top_k, top_p, 0 if do_sample else 1, ops._DT[x.dtype],
                                  torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, lib)
    return out, probs


def _rows(V, dtype, device):
    """A broad row, a peaked one, ties, few finite values, none, NaN, infinity, most of the row equal."""
    g = torch.Generator().manual_seed(V)
    x = torch.randn(10, V, generator=g) * 2.5
    x[1, torch.randperm(V, generator=g)[:40]] += 12
    x[2] = (x[2] * 2).round() / 2
    x[3, torch.randperm(V, generator=g)[:V - 17]] = float("-inf")
    x[4] = float("-inf")
    x[5, V // 2] = float("nan")
    x[6, V - 1] = float("inf")
    x[7] = -1.25
    x[7, ::1000] = 1.0
    x[8, : V // 2] = float("-inf")
    x[9, V - 1] = x[9, 3] = 40.0
    return x.to(dtype).to(device)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V,stride", [(16385, 16385), (16388, 16391), (32769, 32769), (50257, 50257), (98305, 98312), (81923, 81928),
                                      (128255, 128255), (128256, 128256), (262144, 262144), (262145, 262145)])
def test_parts_equal_the_one_launch_kernel(device, V, stride, dtype):
    x = torch.zeros(10, stride, dtype=dtype, device=device)[:, :V]
    x.copy_(_rows(V, dtype, device))
    u = torch.linspace(0.01, 0.99, x.shape[0], device=device)
    calls = [(0.8, 50, 0.9, True), (1.0, 1, 1.0, True), (1.3, 200, 0.95, True), (0.6, 256, 1.0, True),
             (1.0, 257, 0.9, True), (40.0, 20, 0.9, True), (1.0, 0, 1.0, False)]
    assert (_lib.load().aicomp_sample_workspace_bytes(10, V, stride, 0.8, 50, 0, ops._DT[dtype]) > 0) == (V <= 262144)
    for temperature, top_k, top_p, do_sample in calls:
        want, dist = _one_launch(x, temperature, top_k, top_p, do_sample, u)
        got, probs = ops.sample_tokens(x, temperature, top_k, top_p, do_sample, u, return_probs=True)
        plain = ops.sample_tokens(x, temperature, top_k, top_p, do_sample, u)
        assert torch.equal(got, want) and torch.equal(plain, want), (temperature, top_k, top_p)
        assert torch.equal(probs > 0, dist > 0) and torch.allclose(probs, dist, rtol=2.0 ** -22, atol=0.0)


def test_parts_in_a_graph(device):
    x, u = _rows(50257, torch.float32, device), torch.rand(10, device=device)
    ops.sample_tokens(x, 0.8, 50, 0.9, uniforms=u)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        tokens = ops.sample_tokens(x, 0.8, 50, 0.9, uniforms=u)
    for seed in range(3):
        x.copy_(x[torch.randperm(10, device=device)])
        u.uniform_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(tokens, _one_launch(x, 0.8, 50, 0.9, True, u)[0])


@pytest.mark.parametrize("k,room", [(1, 264), (50, 656), (96, 1024), (256, 1024)])
def test_a_part_with_as_many_candidates_as_it_has_room_for(device, k, room):
    """Equal logits on top, as many as one part's list holds and one more (its row then goes the whole way)."""
    V, lib = 131072, _lib.load()
    assert lib.aicomp_sample_workspace_bytes(4, V, V, 1.0, k, 0, _lib.F32) == 4 * 8 * (8 * room + 4)
    x = torch.randn(4, V, generator=torch.Generator().manual_seed(k)).to(device)
    for row, n in enumerate((room - 1, room, room + 1)):
        x[row, 3 * 16384 + 5:3 * 16384 + 5 + n] = 9.0
    u = torch.tensor([0.999, 0.5, 0.25, 0.75], device=device)
    want, dist = _one_launch(x, 1.0, k, 0.9, True, u)
    got, probs = ops.sample_tokens(x, 1.0, k, 0.9, True, u, return_probs=True)
    assert torch.equal(got, want) and torch.equal(probs > 0, dist > 0)
    assert torch.allclose(probs, dist, rtol=2.0 ** -22, atol=0.0)


@pytest.mark.parametrize("k", [1, 15, 16, 17, 63, 64, 65])
@pytest.mark.parametrize("V", [16385, 20000, 50257, 81920, 128256, 262144])
def test_the_short_merge_draws_what_one_launch_draws(device, V, k):
    """Up to 64 kept candidates are drawn from by one wave: k on either side, as many equal logits at the top as its
    lanes and one more, all candidates in one part, fewer finite logits than k, several draws each."""
    x = torch.cat([_rows(V, torch.float32, device), torch.randn(4, V, generator=torch.Generator().manual_seed(k)).to(device)])
    x[10, torch.arange(64, device=device) * (V // 64)] = 9.0
    x[11, torch.arange(65, device=device) * (V // 65)] = 9.0
    x[12, 7:7 + 300] += 20.0
    x[13, 5:] = float("-inf")
    for i in range(6):
        u = torch.rand(x.shape[0], generator=torch.Generator().manual_seed(i)).to(device)
        u[:2] = torch.tensor([0.0, 1.0 - 2.0 ** -24])
        top_p = (1.0, 0.9, 0.5, 0.05, 0.0, 0.999)[i]
        got = ops.sample_tokens(x, 0.7, k, top_p, uniforms=u)
        assert torch.equal(got, _one_launch(x, 0.7, k, top_p, True, u)[0]), (top_p, i)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V,stride,B", [(16385, 16385, 10), (32769, 32776, 10), (50257, 50257, 10), (50256, 50256, 70),
                                        (81921, 81928, 10), (128255, 128255, 10), (128256, 128256, 10),
                                        (262144, 262144, 10), (262145, 262152, 10)])
def test_whole_rows_in_parts(device, V, stride, B, dtype):
    """Draws without top-k: the whole row, and a nucleus of it whose threshold falls among ties, into the largest value, below
    the slices of logits that are looked at (a flat row), or nowhere (no mass).  Masses are whole numbers, so the tokens
    are the same ones."""
    x = torch.zeros(B, stride, dtype=dtype, device=device)[:, :V]
    x.copy_(_rows(V, dtype, device).repeat(B // 10, 1))
    u = torch.rand(B, generator=torch.Generator().manual_seed(V)).to(device)
    u[0], u[1] = 0.0, 1.0 - 2.0 ** -24
    for temperature, top_k, top_p in [(1.0, 0, 1.0), (0.8, V, 1.0), (40.0, 0, 1.0), (0.8, 0, 0.9), (1.0, -1, 0.5), (0.6, 0, 0.95),
                                      (1.3, V, 0.999), (40.0, 0, 0.9), (1.0, 0, 0.0), (0.05, 0, 0.7)]:
        want, _ = _one_launch(x, temperature, top_k, top_p, True, u)
        got = ops.sample_tokens(x, temperature, top_k, top_p, True, u)
        assert torch.equal(got, want), (temperature, top_k, top_p, got, want)


@pytest.mark.parametrize("top_p", [1.0, 0.9])
def test_whole_rows_in_parts_in_a_graph(device, top_p):
    x, u = _rows(81920, torch.float32, device), torch.rand(10, device=device)
    ops.sample_tokens(x, 0.8, 0, top_p, uniforms=u)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = ops.sample_tokens(x, 0.8, 0, top_p, uniforms=u)
    for i in range(3):
        u.copy_(torch.rand(10, device=device))
        x.copy_(x.roll(1, 0))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, _one_launch(x, 0.8, 0, top_p, True, u)[0]), i


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k", [50, 56, 57, 60, 61, 64])
@pytest.mark.parametrize("V", [20000, 81920, 128256])
def test_ties_of_16_bit_rows(device, V, k, dtype):
    """Ties of the k-th value beside it, as many as leave the short merge its 64 lanes and more."""
    x = torch.cat([_rows(V, dtype, device)] * 2)
    for row, n in enumerate((1, 14, 15, 16, 60, 70)):
        x[row, :] = x[row, :].clamp(max=5.0)
        x[row, torch.arange(k - 1, device=device) * 7 + 3] = 9.0
        x[row, V - 1 - torch.arange(n, device=device) * 5] = 8.0
    for i in range(4):
        u = torch.rand(x.shape[0], generator=torch.Generator().manual_seed(i)).to(device)
        top_p = (1.0, 0.9, 0.999, 0.3)[i]
        got = ops.sample_tokens(x, 0.8, k, top_p, uniforms=u)
        assert torch.equal(got, _one_launch(x, 0.8, k, top_p, True, u)[0]), (top_p, i)
