"""Lists and small levels: how many waves share 64 items (32 for rows of 256 columns) goes by items, trees and centroids;
every number of them against exact arithmetic on whole numbers, with last sets of one item."""
import numpy as np
import pytest
import torch

from test_assign_gpu import _blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("trees,n,d,bf", [
    (1, 65, 128, 8),       # 9 centroids: one tile, one wave to 64 items, the second set one item
    (1, 321, 128, 8),      # 41: three tiles
    (3, 1921, 64, 8),      # 241: eight waves to 64 items
    (40, 1025, 128, 8),    # 129: four or fewer
    (60, 1985, 64, 8),     # 249: more sets than waves fit
    (130, 1025, 128, 16),  # 65: one wave to 64 items, from the first round on
    (70, 545, 256, 8),     # 69, sets of 32
    (2, 4161, 64, 8),      # 521: later rounds of the packing walk the full ones too
    (3, 12001, 64, 8),     # 1501: only from the third on
])
def test_waves_that_share_items(trees, n, d, bf, gpu_device):
    from hira_amd.indexer.hip import HIPIndexer

    print(f"case trees={trees} n={n} d={d} bf={bf}", flush=True)
    rng = np.random.default_rng(n + trees)
    x = rng.integers(-4, 5, size=(trees, n, d)).astype(np.float32)
    x[:, 10:60] = x[:, :1]
    keys = torch.from_numpy(x)[None].bfloat16()
    index = HIPIndexer(2, 0, bf, seed=5).build(keys, keys.clone())
    torch.cuda.synchronize()
    K = -(-n // bf)
    for t in sorted({0, trees // 2, trees - 1}):
        want = _blocks(torch.from_numpy(x[t]).to(gpu_device).double(), K, bf, 5 + 7919, t, 8)
        got = index.perm[t, :K * bf].cpu().numpy().reshape(K, bf)
        np.testing.assert_array_equal(got, want, err_msg=f"tree {t}")
