"""Draws from a list of candidates: as many as the kernels rank at once and one more, in one launch and from a row's parts."""
import numpy as np
import pytest
import torch

from aicomp_amd import _lib, ops
from oracle import sample_oracle as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [16384, 131072])
@pytest.mark.parametrize("n", [1, 63, 65, 127, 128, 129, 256, 257, 384, 385, 512, 513, 1000, 1024, 1025])
def test_equal_logits_are_drawn_in_index_order(device, V, n):
    """n equal logits on top, all of them kept: equal masses, so the draw is the floor(u n)-th of them, and half of the mass
    keeps the first n // 2 + 1.  u over multiples of 1/64 (odd ones beside the steps), products exact in double."""
    k = min(n, 100)
    assert (_lib.load().aicomp_sample_workspace_bytes(32, V, V, 0.8, k, 0, _lib.F32) > 0) == (V > 16384)
    g = torch.Generator().manual_seed(n)
    x = torch.randn(32, V, generator=g)
    at = torch.stack([torch.randperm(V, generator=g)[:n].sort().values for _ in range(32)])
    x.scatter_(1, at, 40.0)
    u = (torch.arange(32) * 2 + 1) / 64
    for top_p, kept in ((1.0, n), (0.5, n // 2 + 1)):
        tokens = ops.sample_tokens(x.to(device), 0.8, k, top_p, uniforms=u.to(device)).cpu()
        assert torch.equal(tokens, at.gather(1, (u.double() * kept).long()[:, None])[:, 0]), top_p


@pytest.mark.parametrize("dtype,name", [(torch.float32, "f32"), (torch.bfloat16, "bf16"), (torch.float16, "f16")])
@pytest.mark.parametrize("V,k", [(20000, 65), (20000, 129), (20000, 300), (20000, 700), (40000, 90), (65536, 100), (131072, 66), (131072, 130),
                                 (131072, 200), (131072, 256), (262144, 256)])
def test_lists_of_distinct_logits(device, V, k, dtype, name):
    """Kept set, masses and the inverse CDF in index order against the oracle.  A mass is rounded to 2^-40 of the largest, its
    exponential to a few 2^-24: 2e-5 of each, 1e-6 of a sum."""
    g = torch.Generator().manual_seed(V + k)
    x = (torch.randn(3, V, generator=g) * 2.5).to(dtype)
    x[1, torch.randperm(V, generator=g)[:k // 2]] += 9
    x[2, V // 3:V // 3 + k] += 9
    u = torch.rand(3, generator=g)
    check_draws(device, x, u, k, name)


@pytest.mark.parametrize("dtype,name", [(torch.float32, "f32"), (torch.bfloat16, "bf16")])
@pytest.mark.parametrize("V,k", [(40000, 65), (131072, 50), (131072, 65), (131072, 100), (131072, 256), (262144, 64), (262144, 200)])
def test_lists_of_clustered_logits(device, V, k, dtype, name):
    """Rows whose top is in few parts, or in few waves of a part: likelier tokens of lower index, as a language model's (lists longer
    than their room at first, k 256), all of it in the last part but one, and clusters of 256 (rows done whole)."""
    g = torch.Generator().manual_seed(V + k)
    fall = torch.log1p(torch.arange(V, dtype=torch.float32))
    x = torch.randn(5, V, generator=g)
    x[0] = x[0] * 1.5 - fall
    x[1] -= fall
    x[2] = x[2] * 2.5 - 2 * fall
    part = 16384 * ((V - 1) // 16384 - 1)
    x[3, part + torch.randperm(16384, generator=g)[:2 * k]] += 30
    x[4] += torch.randn((V + 255) // 256, generator=g).mul(2).repeat_interleave(256)[:V]
    check_draws(device, x.to(dtype), torch.rand(5, generator=g), k, name)


def check_draws(device, x, u, k, name):
    for top_p in (1.0, 0.9):
        tokens, probs = ops.sample_tokens(x.to(device), 0.8, k, top_p, uniforms=u.to(device), return_probs=True)
        plain = ops.sample_tokens(x.to(device), 0.8, k, top_p, uniforms=u.to(device))
        assert torch.equal(plain, tokens)
        for b in range(len(x)):
            row, p = x[b].float().numpy(), probs[b].cpu().double().numpy()
            want = S.filtered_probs(row, 0.8, k, top_p, name)
            if top_p < 1:                                   # entries at the threshold may fall on either side
                sure = S.nucleus_margin(row, 0.8, k, top_p, name) > 2e-5
                assert np.array_equal((p > 0)[sure], (want > 0)[sure])
            else:
                assert np.array_equal(p > 0, want > 0)
            if np.array_equal(p > 0, want > 0):
                assert np.allclose(p, want, rtol=2e-5, atol=1e-9)
            cdf, t = np.cumsum(p), int(tokens[b])
            assert p[t] > 0 and cdf[t] - p[t] - 1e-6 <= float(u[b]) <= cdf[t] + 1e-6
