"""Levels of few items, which one launch takes as a whole, against the launches that take the larger
ones: a build that is given the trees' key counts goes through those whatever its size, and clusters the
same keys into the same blocks.  Bit for bit, over ties, buckets far larger than a block, keys that are
no numbers, and sizes around the kernel's stretches (64 lanes, 32 centroids, 16384 pairs, 1024 items)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _keys(kind, h, n, d, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    k = torch.randn(1, h, n, d, generator=g, device="cuda")
    if kind == "ties":  # every row several times
        k = k[:, :, torch.arange(n, device="cuda") % max(1, n // 5)]
    if kind == "hub":   # most rows close to one of them
        k = torch.where(torch.arange(n, device="cuda")[:, None] % 7 > 0, 3.0 + 0.01 * k, k)
    if kind == "nan":
        k[:, :, ::11, 1] = float("nan")
        k[:, :, ::17, 2] = float("inf")
    return k.to(torch.bfloat16).contiguous()


def _arrays(idx):
    return [idx.perm, idx.keys_buf.view(torch.int16), idx.values_buf.view(torch.int16), idx.counts[1],
            idx.centers[1].view(torch.int16), idx.radii[1].view(torch.int32)]


@pytest.mark.parametrize("kind", ["normal", "ties", "hub", "nan"])
@pytest.mark.parametrize("h,n,d,bf,niter", [(1, 1, 128, 32, 1), (2, 2, 64, 2, 0), (3, 63, 128, 16, 1), (2, 65, 64, 64, 2),
                                            (1, 32, 64, 1, 1), (2, 500, 256, 32, 1), (2, 510, 256, 16, 1),
                                            (3, 1000, 64, 64, 2), (8, 512, 128, 16, 1), (2, 511, 128, 17, 1),
                                            (2, 513, 128, 17, 1), (1, 1024, 128, 64, 3), (1, 1025, 128, 64, 1)])
def test_a_small_level_is_clustered_as_a_large_one(kind, h, n, d, bf, niter, gpu_device):
    from hira_amd.indexer import HIPIndexer

    keys, vals = _keys(kind, h, n, d, n), _keys("normal", h, n, d, n + 1)
    one = HIPIndexer(2, niter, bf).build(keys, vals)
    many = HIPIndexer(2, niter, bf).build(keys, vals, key_counts=torch.full((h,), n, dtype=torch.int32, device="cuda"))
    for a, b in zip(_arrays(one), _arrays(many)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("h,n,d,levels,bf", [(2, 1111, 64, 5, 10), (3, 8192, 128, 3, 32), (1, 700, 128, 4, 5)])
def test_levels_above_cluster_the_centres_below(h, n, d, levels, bf, gpu_device):
    """Every level holds each node of the level below once, at most bf a block, and its centre is their
    mean: the launch goes on to the levels above by itself."""
    from hira_amd.indexer import HIPIndexer
    from hira_amd.indexer.hip import from_tiled

    idx = HIPIndexer(levels, 1, bf).build(_keys("normal", h, n, d, 5), _keys("normal", h, n, d, 6))
    perm = idx.perm[:, : idx.size[0]]
    for t in range(h):
        p = perm[t][perm[t] >= 0]
        assert torch.equal(p.sort().values, torch.arange(n, device="cuda", dtype=p.dtype))
    rows = lambda x, tiled: (from_tiled(x) if tiled else x).float()
    for l in range(2, levels):
        cnt, below = idx.counts[l][:, : idx.size[l]], idx.counts[l - 1][:, : idx.size[l - 1]]
        assert int(cnt.max()) <= bf and bool((cnt.sum(1) == (below > 0).sum(1)).all())
        child, centre = rows(idx.centers[l - 1], idx.tiled), rows(idx.centers[l], idx.tiled)
        for t in range(h):
            for k in range(idx.size[l]):
                c = int(cnt[t, k])
                if c:
                    mean = child[t, k * bf: k * bf + c].mean(0)
                    # (one rounding to bf16, 2^-9 of a number, and fp32 sums)
                    assert torch.allclose(centre[t, k], mean, rtol=2 ** -8, atol=1e-5)


@pytest.mark.parametrize("kind", ["normal", "hub"])
@pytest.mark.parametrize("h,n,d,bf,niter", [(1, 1024, 128, 32, 1), (2, 1023, 64, 32, 2), (1, 993, 128, 32, 0), (1, 512, 256, 32, 1),
                                            (2, 97, 128, 3, 1), (2, 1009, 128, 32, 1)])
def test_as_many_pairs_as_the_scores_have_room_for(kind, h, n, d, bf, niter, gpu_device):
    test_a_small_level_is_clustered_as_a_large_one(kind, h, n, d, bf, niter, gpu_device)


@pytest.mark.parametrize("kind", ["normal", "ties", "hub", "nan"])
@pytest.mark.parametrize("h,n,d,bf", [(2, 16, 64, 8), (2, 255, 128, 16), (2, 256, 64, 32), (2, 257, 128, 16), (1, 512, 64, 64),
                                      (2, 513, 64, 32), (1, 769, 128, 64), (2, 264, 256, 33)])
def test_item_tiles_of_a_wave(kind, h, n, d, bf, gpu_device):
    """Around 256 and 512 items a wave holds one, two or four of the tiles of sixteen."""
    test_a_small_level_is_clustered_as_a_large_one(kind, h, n, d, bf, 2, gpu_device)
