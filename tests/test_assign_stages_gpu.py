"""The approximate assignment walks the centroids in stages of eight tiles of 16 (four for rows of 256 columns),
of arrays padded to four: numbers of centroids whose last stage is half there, has one tile, or is
whole, for all of them and for those with room only, against exact arithmetic on whole numbers."""
import numpy as np
import pytest
import torch

from test_assign_gpu import _blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,trees,K,d,bf", [
    (torch.bfloat16, 2, 256, 128, 8),      # whole stages
    (torch.bfloat16, 2, 257, 128, 8),      # 20 tiles: half a stage at the end, one column of it in use
    (torch.bfloat16, 2, 320, 64, 8),       # 20 tiles, all of them in use
    (torch.bfloat16, 1, 321, 256, 8),      # 24 tiles: six stages of four
    (torch.bfloat16, 1, 273, 256, 16),     # 20 tiles
    (torch.bfloat16, 9, 520, 128, 16),     # 36 tiles; lists long enough for the approximate pass
    (torch.float32, 1, 48, 36, 32),        # 4 tiles: half a stage is all there is
    (torch.float32, 2, 65, 100, 16),       # 8 tiles
    (torch.float32, 1, 577, 256, 8),
])
def test_last_stage(dtype, trees, K, d, bf, gpu_device):
    from hira_amd.indexer.hip import HIPIndexer

    n = K * bf - 3
    print(f"case {dtype} trees={trees} K={K} n={n} d={d} bf={bf}", flush=True)
    rng = np.random.default_rng(K + d)
    x = rng.integers(-4, 5, size=(trees, n, d)).astype(np.float32)
    x[:, n // 3:n // 3 + 40] = x[:, -1:]  # the last centroid's bucket overflows
    keys = torch.from_numpy(x)[None].to(dtype)
    index = HIPIndexer(2, 0, bf, seed=5).build(keys, keys.clone())
    torch.cuda.synchronize()
    for t in range(trees):
        want = _blocks(torch.from_numpy(x[t]).to(gpu_device).double(), K, bf, 5 + 7919, t, 8)
        got = index.perm[t, :K * bf].cpu().numpy().reshape(K, bf)
        np.testing.assert_array_equal(got, want, err_msg=f"tree {t}")
