"""Float32 prefill where waves share query rows and split the keys (small grids): every row against the
float64 oracle, on either side of the lines and of the tiles' edges."""
import pytest
import torch

from helpers import to_f64
from test_gpu_prefill import build_case, oracle, run

pytestmark = pytest.mark.gpu

# (waves per row, priors, chunks, query heads, KV heads): workgroups of 128 rows = heads / group packed x tiles
SHAPES = [(4, [0, 7, 61], [1, 33, 130], 8, 2), (4, [15, 16, 17, 0], [17, 16, 15, 64], 16, 16),
          (4, [300, 1], [2, 127], 16, 1), (4, [63, 64, 65], [1, 1, 129], 6, 2),
          (2, [0, 31, 32, 33, 200, 5], [1, 32, 31, 65, 40, 128], 32, 32),
          (1, [9 * i for i in range(14)], [1 + 3 * i for i in range(14)], 32, 32)]


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("kw,priors,news,hq,hkv", SHAPES)
def test_rows_shared_by_waves(device, kw, priors, news, hq, hkv, d):
    group = hq // hkv
    gpack = group if 16 % group == 0 else 1
    tiles = -(-max(news) // (128 // gpack)) * len(news)
    wgs = hq // gpack * min(tiles, sum(news) // (128 // gpack) + len(news))
    assert kw == (4 if wgs <= 128 else 2 if wgs <= 400 else 1)
    c = build_case(device, priors, news, hq, hkv, d, dtype=torch.float32, seed=kw + d, poison="all")
    err = abs(to_f64(run(c, max_q_len=max(news))) - oracle(c)).max()
    assert err <= 1e-5, err                                # float32 sums of at most 430 keys of N(0, 1/4)
