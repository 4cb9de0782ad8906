"""The index build's nearest-centroid assignment and packing against the same steps in exact integer
arithmetic: keys of small whole numbers, initial centroids taken as they are (no Lloyd round), so
every distance is exact in any order of summation and ties are many.  Sizes around the numbers of
centroids and items at which another kernel takes over, and rows of every width class."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

M64 = (1 << 64) - 1


def _mix64(z):
    z = (z + 0x9E3779B97F4A7C15) & M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
    return z ^ (z >> 31)


def _blocks(x, K, bf, seed, tree, rounds):
    """Slots (K, bf) of one tree: seeds, then `rounds` of proposals, then what is left in order."""
    n = x.shape[0]
    seeds = []
    for k in range(K):
        u = float(_mix64(seed ^ _mix64((tree * 0x100000001B3 + k) & M64)) >> 11) / 9007199254740992.0
        seeds.append(min(int((k + u) * n / K), n - 1))
    c = x[seeds]
    d2 = ((x * x).sum(1, keepdim=True) + (c * c).sum(1)[None] - 2.0 * (x @ c.t().contiguous())) * K
    d2 += torch.arange(K, device=x.device, dtype=torch.float64)  # (whole numbers: lowest centroid on ties)
    slots, fill = np.full((K, bf), -1, np.int64), np.zeros(K, np.int64)
    todo = np.arange(n)
    for _ in range(rounds):
        if len(todo) == 0:
            break
        full = torch.from_numpy(fill >= bf).to(x.device)
        d = d2[torch.from_numpy(todo).to(x.device)].masked_fill(full[None], float("inf")).min(1).values.cpu().numpy()
        k, dist = (d % K).astype(np.int64), d // K
        order = np.lexsort((todo, dist, k))
        k, items = k[order], todo[order]
        place = np.arange(len(k)) - np.searchsorted(k, k)  # rank among the proposers of its centroid
        ok = place < bf - fill[k]
        slots[k[ok], (fill[k] + place)[ok]] = items[ok]
        fill += np.bincount(k[ok], minlength=K)
        todo = np.sort(items[~ok])
    free = [(k, j) for k in range(K) for j in range(fill[k], bf)] if len(todo) else []
    for i, (k, j) in zip(todo, free):
        slots[k, j] = i
    return slots


@pytest.mark.parametrize("dtype,trees,n,d,bf,values", [
    (torch.bfloat16, 2, 2040, 128, 8, 4),      # 255 centroids: both halves at once
    (torch.bfloat16, 2, 2043, 128, 8, 4),      # 256: the approximate pass, a ragged last block
    (torch.bfloat16, 3, 5000, 64, 16, 2),      # 313, few values: ties and items it is unsure of
    (torch.bfloat16, 1, 9001, 256, 32, 3),
    (torch.bfloat16, 2, 1535, 96, 32, 4),      # 48: no exact kernel on the matrix cores for this width
    (torch.bfloat16, 2, 3001, 40, 16, 3),
    (torch.float32, 2, 1503, 36, 32, 3),       # 47: the vector kernel alone
    (torch.float32, 2, 1505, 36, 32, 3),       # 48
    (torch.float32, 1, 4100, 256, 8, 4),       # 513: lists against the centroids with room only
    (torch.bfloat16, 8, 33000, 128, 64, 6),    # 516, and lists long enough for the approximate pass
])
def test_blocks_equal_exact_arithmetic(dtype, trees, n, d, bf, values, gpu_device):
    from hira_amd.indexer.hip import HIPIndexer

    print(f"case {dtype} trees={trees} n={n} d={d} bf={bf}", flush=True)
    rng = np.random.default_rng(n + d)
    x = rng.integers(-values, values + 1, size=(trees, n, d)).astype(np.float32)
    x[:, n // 2:n // 2 + 300] = x[:, :1]  # a bucket beyond what the members' array holds
    keys = torch.from_numpy(x)[None].to(dtype)
    index = HIPIndexer(2, 0, bf, seed=5).build(keys, keys.clone())
    torch.cuda.synchronize()
    K = -(-n // bf)
    for t in range(trees):
        want = _blocks(torch.from_numpy(x[t]).to(gpu_device).double(), K, bf, 5 + 7919, t, 8)
        got = index.perm[t, :K * bf].cpu().numpy().reshape(K, bf)
        np.testing.assert_array_equal(got, want, err_msg=f"tree {t}")


@pytest.mark.parametrize("dtype,n,d,bf", [(torch.bfloat16, 3000, 128, 8), (torch.float32, 700, 36, 16)])
def test_keys_that_are_no_numbers_keep_a_slot(dtype, n, d, bf, gpu_device):
    from hira_amd.indexer.hip import HIPIndexer

    x = torch.randn(1, 2, n, d, generator=torch.Generator().manual_seed(n))
    x[:, :, 5::97, 3] = float("nan")
    index = HIPIndexer(2, 1, bf, seed=2).build(x.to(dtype), x.to(dtype))
    perm = index.perm[:, :-(-n // bf) * bf].cpu().numpy()
    for t in range(2):
        assert sorted(perm[t][perm[t] >= 0].tolist()) == list(range(n))


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.float32, 36)])
@pytest.mark.parametrize("bf,places", [(1, 64), (4, 64), (5, 128), (8, 128), (9, 256), (32, 256), (64, 256)])
@pytest.mark.parametrize("more", [-1, 0, 1, 3])
def test_buckets_around_the_places_they_have(dtype, d, bf, places, more, gpu_device):
    """The largest bucket one item below, at and beyond the places that a fan-out gives each."""
    from hira_amd.indexer.hip import HIPIndexer

    n = 70 * bf + 400
    rng = np.random.default_rng(bf)
    x = rng.integers(-4, 5, size=(1, n, d)).astype(np.float32)
    x[:, 1:places + more] = x[:, :1]  # (row 0 is the first centroid)
    keys = torch.from_numpy(x)[None].to(dtype)
    index = HIPIndexer(2, 0, bf, seed=5).build(keys, keys.clone())
    K = -(-n // bf)
    want = _blocks(torch.from_numpy(x[0]).to(gpu_device).double(), K, bf, 5 + 7919, 0, 8)
    np.testing.assert_array_equal(index.perm[0, :K * bf].cpu().numpy().reshape(K, bf), want)
    # with Lloyd rounds: means over the same buckets, in a fixed order
    a, b = (HIPIndexer(2, 2, bf, seed=5).build(keys, keys.clone()) for _ in range(2))
    assert torch.equal(a.perm, b.perm) and torch.equal(a.radii[1], b.radii[1])
    assert sorted(a.perm[a.perm >= 0].tolist()) == list(range(n))
