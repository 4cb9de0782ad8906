"""Sample thresholds from bf16 rows of 64 and 128 columns: numbers of samples around the rows of a pass (128, 64)
and of a round (1024), where the last pass is moved back and scores rows that another one has, and k around
the sixteen that a merge keeps."""
import numpy as np
import pytest
import torch

from oracle import hira_oracle as ho
from helpers import bf16_round, clustered_keys, random_query

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("s", [1, 2, 63, 64, 65, 127, 128, 129, 191, 960, 1000, 1023, 1024, 1025, 1100, 2049, 4095])
def test_every_row_counts_once(s, d, gpu_device):
    from hira_amd.cache import threshold_finder as tf

    print(f"case s={s} d={d}", flush=True)
    t, h = 2, 6
    x = bf16_round(clustered_keys(t, s, d, seed=3 + s, clusters=max(1, s // 40)))
    q = bf16_round(random_query(h, d, seed=11 + s))
    xd, qd = torch.from_numpy(x).bfloat16().cuda(), torch.from_numpy(q).bfloat16().cuda()
    scale = float(np.abs(ho.sample_thresholds(x, q, "sample_max")).max()) + 1e-6
    got = tf.sample_max(xd, qd).cpu().numpy()
    assert np.abs(got - ho.sample_thresholds(x, q, "sample_max")).max() <= 1e-5 * scale
    for k in sorted({1, min(s, 10), min(s, 15), min(s, 16), min(s, 17), s}):
        got = tf.sample_mean_topk(xd, qd, k).cpu().numpy()
        # fp32 sums of d products and of k scores
        assert np.abs(got - ho.sample_thresholds(x, q, "sample_mean_topk", k)).max() <= 1e-5 * scale, k
        if k == 1:
            assert np.array_equal(got, tf.sample_max(xd, qd).cpu().numpy())


def test_equal_scores(gpu_device):
    """Ties among the best: as many of them as k asks for count."""
    from hira_amd.cache import threshold_finder as tf

    x = torch.ones(1, 700, 128).bfloat16()
    x[:, 5::9] = 2.0  # 78 rows
    q = torch.ones(2, 128).bfloat16()
    for k in (1, 16, 77, 79):
        got = tf.sample_mean_topk(x.cuda(), q.cuda(), k).cpu()
        want = 128.0 * (2.0 * min(k, 78) + max(k - 78, 0)) / k
        assert torch.allclose(got, torch.full((2,), want), rtol=1e-6)


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 8), (torch.bfloat16, 16), (torch.float32, 4), (torch.float32, 8)])
def test_the_best_member_of_a_sample_is_selected(dtype, d, gpu_device):
    """Rows of one or two chunks score the same in the threshold and in the search: under a sample's maximum the
    key that makes the threshold is selected."""
    from hira_amd.cache import threshold_finder as tf
    from hira_amd.indexer import HIPIndexer
    from hira_amd.searcher import HIPSearcher

    g = torch.Generator().manual_seed(d)
    keys = torch.randn(1, 8, 900, d, generator=g).to(dtype).cuda()
    index, searcher = HIPIndexer(2, 1, 16).build(keys), HIPSearcher(output_fill_value=float("-inf"))
    for _ in range(8):
        q = torch.randn(64, d, generator=g).to(dtype).cuda()
        tau = tf.sample_max(keys[0], q)
        assert torch.equal(tau, tf.sample_mean_topk(keys[0], q, 1))
        assert torch.equal(searcher.search(q, tau, index).amax(dim=1), tau)
