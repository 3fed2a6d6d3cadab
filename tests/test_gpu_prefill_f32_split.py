"""Float32 prefill where waves share query rows and split the keys (small grids): every row against the
float64 oracle, on either side of the lines and of the tiles' edges."""
import pytest
import torch

from helpers import kernels_of, to_f64
from test_gpu_prefill import build_case, oracle, run

pytestmark = pytest.mark.gpu

# (waves per row of the kernel that is to run, priors, chunks, query heads, KV heads)
SHAPES = [(4, [0, 7, 61], [1, 33, 130], 8, 2), (4, [15, 16, 17, 0], [17, 16, 15, 64], 16, 16),
          (4, [300, 1], [2, 127], 16, 1), (4, [63, 64, 65], [1, 1, 129], 6, 2),
          (2, [0, 31, 32, 33, 200, 5], [1, 32, 31, 65, 40, 128], 32, 32),
          (1, [9 * i for i in range(14)], [1 + 3 * i for i in range(14)], 32, 32),
          # many chunks: four waves per row, then two, would be more workgroups than CUs
          (2, [0, 5, 64, 31, 1, 0, 90, 16], [46, 24, 33, 1, 17, 46, 40, 8], 32, 8),
          (1, [0, 3, 64, 31, 0, 0, 90, 16], [70, 66, 64, 65, 70, 63, 67, 70], 32, 8)]


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("kw,priors,news,hq,hkv", SHAPES)
def test_rows_shared_by_waves(device, kw, priors, news, hq, hkv, d):
    c = build_case(device, priors, news, hq, hkv, d, dtype=torch.float32, seed=kw + d, poison="all")
    outs = []
    names = kernels_of(lambda: outs.append(run(c, max_q_len=max(news))))
    assert any(f"paged_prefill_mfma_f32_kernel<{d}, {kw}>" in n for n in names), names
    err = abs(to_f64(outs[0]) - oracle(c)).max()
    assert err <= 1e-5, err                                # float32 sums of at most 430 keys of N(0, 1/4)
