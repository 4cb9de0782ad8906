"""Windows of new keys that open nodes, on trees whose level-2 nodes have room here and there, against the same keys
one by one: up to, at and beyond what the list of parents holds, ties between parents, no room left, three and four
levels, a key that has no finite distance to any parent."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _full_below(trees, k2, levels, bf, d, dtype, seed):
    """Level-1 nodes are full; level-2 node q has 1 .. bf of them (q = 0 and 1 share a centre); one root above for four."""
    rng = np.random.default_rng(seed)
    k1, n = k2 * bf, k2 * bf * bf

    def rnd(x):
        return torch.from_numpy(x.astype(np.float32)).to(dtype).float().numpy()

    counts2 = np.tile(rng.integers(1, bf, size=k2), (trees, 1)).astype(np.int32)
    c2 = rnd(rng.normal(size=(trees, k2, d)))
    if k2 > 1:
        c2[:, 1] = c2[:, 0]
    c1 = rnd(np.repeat(c2, bf, axis=1) + 0.2 * rng.normal(size=(trees, k1, d)))
    keys = rnd(np.repeat(c1, bf, axis=1) + 0.1 * rng.normal(size=(trees, n, d)))
    used1 = (np.arange(bf)[None, None] < counts2[:, :, None]).reshape(trees, k1)
    used0 = np.repeat(used1, bf, axis=1)
    c1[~used1], keys[~used0] = 0, 0
    perm = np.full((trees, n), -1, np.int32)
    for t in range(trees):
        perm[t, used0[t]] = np.arange(used0[t].sum())
    r1 = np.linalg.norm(keys - np.repeat(c1, bf, axis=1), axis=2).reshape(trees, k1, bf).max(2) * 1.0001
    r1[~used1] = -np.inf
    need = np.linalg.norm(c1 - np.repeat(c2, bf, axis=1), axis=2) + r1
    r2 = need.reshape(trees, k2, bf).max(2) * 1.0001
    counts1 = np.where(used1, bf, 0).astype(np.int32)
    centers, radii, counts = [None, c1, c2], [None, r1, r2], [None, counts1, counts2]
    if levels == 4:
        c3 = rnd(c2.mean(1, keepdims=True))
        centers.append(c3)
        radii.append((np.linalg.norm(c2 - c3, axis=2) + r2).max(1, keepdims=True) * 1.0001)
        counts.append(np.full((trees, 1), k2, np.int32))
    return dict(bf=bf, keys=keys, values=keys.copy(), perm=perm, centers=centers, radii=[None] + [r.astype(np.float32) for r in radii[1:]],
                counts=counts, dtype=dtype), int(used0[0].sum())


@pytest.mark.parametrize("k2,levels,bf,m,d,dtype,layout,bad", [
    (1, 3, 4, 70, 64, torch.float32, "row_major", None),      # few places: then new nodes of level 2
    (16, 3, 8, 64, 128, torch.float32, "row_major", None),    # as many as the list holds in fp32
    (17, 3, 8, 40, 128, torch.float32, "row_major", None),    # one more
    (32, 3, 4, 130, 256, torch.bfloat16, "row_major", None),  # as many as it holds in bf16, chunks of keys
    (33, 3, 4, 64, 64, torch.bfloat16, "row_major", None),
    (16, 4, 16, 200, 128, torch.bfloat16, "tiled", None),     # a level above
    (3, 3, 16, 64, 128, torch.bfloat16, "q8", None),
    (3, 3, 16, 64, 64, torch.bfloat16, "q8", None),
    (4, 3, 4, 64, 128, torch.bfloat16, "row_major", {0: "huge", 33: "nan"}),
])
def test_a_window_that_opens_nodes_equals_key_by_key(k2, levels, bf, m, d, dtype, layout, bad, gpu_device):
    from hira_amd.indexer.hip import HIPIndexer

    parts, held = _full_below(2, k2, levels, bf, d, dtype, seed=m)
    rng = np.random.default_rng(m)
    c2 = parts["centers"][2]
    pick = rng.integers(0, k2, size=(2, m))
    new = np.stack([c2[t, pick[t]] + 0.3 * rng.normal(size=(m, d)) for t in range(2)]).astype(np.float32)
    new[:, 2::7] = c2[:, :1]  # as near to node 0 as to node 1
    for i, what in (bad or {}).items():
        new[:, i, 3] = {"nan": np.nan, "huge": 3e38}[what]
    N = torch.from_numpy(new)[None].to(dtype).cuda()
    a, b = (HIPIndexer.from_layout(layout=layout, num_keys=held, **parts) for _ in range(2))
    a.graft_min = b.graft_min = 1 << 30
    a.update(N, N)
    for i in range(m):
        b.update(N[:, :, i:i + 1], N[:, :, i:i + 1])
    assert a.size == b.size
    n = a.size[0]

    def same(x, y):  # (a centre or a radius may be no number)
        return torch.equal(torch.nan_to_num(x.float(), nan=1.25e30), torch.nan_to_num(y.float(), nan=1.25e30))

    assert torch.equal(a.perm[:, :n], b.perm[:, :n])
    assert same(a.keys_buf[:, :n // 16 * 16], b.keys_buf[:, :n // 16 * 16])
    assert same(a.values_buf[:, :n], b.values_buf[:, :n])
    for l in range(1, levels):
        k = a.size[l]
        assert torch.equal(a.counts[l][:, :k], b.counts[l][:, :k]), l
        assert same(a.radii[l][:, :k], b.radii[l][:, :k]), l
        assert same(a.centers_rowmajor(l)[:, :k], b.centers_rowmajor(l)[:, :k]), l
    if layout == "q8":
        assert torch.equal(a.keys8[:, :n], b.keys8[:, :n])
        assert torch.equal(a.keps[:, :a.size[1]], b.keps[:, :b.size[1]])
