"""Nearest centroids on the vector units: how many waves share a set of items goes by items, trees and centroids; every
number of them against exact arithmetic on whole numbers, with last sets of one item and waves without a centroid."""
import numpy as np
import pytest
import torch

from test_assign_gpu import _blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,trees,n,d,bf", [
    (torch.float32, 1, 17, 36, 4),       # 5 centroids for eight waves, sets of 16 items
    (torch.float32, 3, 2801, 36, 64),    # 44: eight waves to a set
    (torch.float32, 5, 2801, 36, 64),    # four
    (torch.float32, 6, 2801, 36, 64),    # two
    (torch.float32, 12, 2801, 36, 64),   # one
    (torch.float32, 40, 2801, 36, 64),   # more sets than waves, in strides
    (torch.float32, 2, 1029, 256, 32),   # 33: sets of four
    (torch.bfloat16, 2, 257, 8, 8),      # 33: sets of 128
    (torch.bfloat16, 1, 1440, 40, 32),   # 45
    (torch.float32, 2, 4999, 36, 8),     # 625: more than 64 centroids a wave; lists, and what the approximate pass leaves
])
def test_waves_that_share_items(dtype, trees, n, d, bf, gpu_device):
    from hira_amd.indexer.hip import HIPIndexer

    print(f"case {dtype} trees={trees} n={n} d={d} bf={bf}", flush=True)
    rng = np.random.default_rng(n + trees)
    x = rng.integers(-3, 4, size=(trees, n, d)).astype(np.float32)
    x[:, n // 2:n // 2 + n // 8] = x[:, :1]
    keys = torch.from_numpy(x)[None].to(dtype)
    index = HIPIndexer(2, 0, bf, seed=5).build(keys, keys.clone())
    torch.cuda.synchronize()
    K = -(-n // bf)
    for t in sorted({0, trees // 2, trees - 1}):
        want = _blocks(torch.from_numpy(x[t]).to(gpu_device).double(), K, bf, 5 + 7919, t, 8)
        got = index.perm[t, :K * bf].cpu().numpy().reshape(K, bf)
        np.testing.assert_array_equal(got, want, err_msg=f"tree {t}")
