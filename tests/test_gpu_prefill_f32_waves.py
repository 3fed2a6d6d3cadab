"""Float32 prefill at the edges of its 16-row waves, 128-row workgroups and 32-token tiles, against the
float64 oracle; slots beyond every context are NaN (K) and Inf (V)."""
import numpy as np
import pytest
import torch

from helpers import to_f64
from test_gpu_prefill import build_case, oracle, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,hkv", [(8, 2), (4, 4), (6, 2)])        # 4, 16 and 16 positions per wave
def test_float32_prefill_edges(device, d, hq, hkv):
    news = [1, 3, 4, 5, 15, 16, 17, 31, 32, 33, 65, 127, 129]
    priors = [0, 14, 15, 16, 17, 31, 0, 33, 64, 30, 1, 47, 95]
    c = build_case(device, priors, news, hq, hkv, d, dtype=torch.float32, seed=d + hq, poison="all")
    # the bound of the other float32 prefill tests: a typical error of sqrt(128) 2^-24 a score, outputs of order 1,
    # with a factor of ten
    np.testing.assert_allclose(to_f64(run(c, max(news))), oracle(c), rtol=0, atol=1e-5)
