"""Windows of new keys placed from the list of nodes with room against the same keys one by one, on
trees that have many such nodes: lists of eight and more, up to and beyond what the list holds,
exact ties between nodes, windows beyond 64 keys, wide rows."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _half_full(trees, k2, bf, d, dtype, seed):
    """Three levels, k2 roots, every level-1 node with 1 .. bf keys; node 1's centre equals node 0's."""
    rng = np.random.default_rng(seed)
    k1, n = k2 * bf, k2 * bf * bf

    def rnd(x):
        return torch.from_numpy(x.astype(np.float32)).to(dtype).float().numpy()

    keys, perm = np.zeros((trees, n, d), np.float32), np.full((trees, n), -1, np.int32)
    c1, c2 = rnd(rng.normal(size=(trees, k1, d))), rnd(rng.normal(size=(trees, k2, d)) * 0.1)
    c1[:, 1] = c1[:, 0]
    counts = rng.integers(1, bf + 1, size=(trees, k1)).astype(np.int32)
    counts[:, :2] = 1
    r1, r2 = np.zeros((trees, k1), np.float32), np.zeros((trees, k2), np.float32)
    for t in range(trees):
        at = 0
        for p in range(k1):
            for j in range(counts[t, p]):
                keys[t, p * bf + j] = rnd(c1[t, p] + 0.3 * rng.normal(size=d))
                perm[t, p * bf + j], at = at, at + 1
            r1[t, p] = max(np.linalg.norm(keys[t, p * bf + j] - c1[t, p]) for j in range(counts[t, p])) * 1.0001
        for q in range(k2):
            r2[t, q] = max(np.linalg.norm(c1[t, p] - c2[t, q]) + r1[t, p] for p in range(q * bf, (q + 1) * bf)) * 1.0001
    full = np.full((trees, k2), bf, np.int32)
    return dict(bf=bf, keys=keys, perm=perm, centers=[None, c1, c2], radii=[None, r1, r2], counts=[None, counts, full],
                values=keys.copy(), dtype=dtype), counts.sum(1)


@pytest.mark.parametrize("k2,bf,m,d,dtype,layout", [
    (1, 8, 40, 64, torch.float32, "row_major"),      # a list of up to eight
    (3, 8, 64, 128, torch.bfloat16, "row_major"),    # three eights
    (3, 16, 65, 128, torch.bfloat16, "tiled"),       # up to all 48
    (2, 32, 200, 64, torch.bfloat16, "tiled"),       # more than the list holds
    (3, 8, 130, 256, torch.float32, "row_major"),    # the widest rows, three chunks of keys
    (1, 16, 255, 128, torch.bfloat16, "q8"),
])
def test_window_equals_key_by_key_on_half_full_trees(k2, bf, m, d, dtype, layout, gpu_device):
    from hira_amd.indexer.hip import HIPIndexer

    parts, held = _half_full(2, k2, bf, d, dtype, seed=m)
    # (the trees must hold the same number of keys: the fuller one's last keys are taken out again)
    for t in range(2):
        extra = int(held[t] - held.min())
        while extra:
            node = int(parts["counts"][1][t, 2:].argmax()) + 2
            slot = node * bf + int(parts["counts"][1][t, node]) - 1
            gone = parts["perm"][t, slot]
            parts["perm"][t][parts["perm"][t] > gone] -= 1
            parts["perm"][t, slot], parts["keys"][t, slot] = -1, 0
            parts["counts"][1][t, node] -= 1
            extra -= 1
    parts["values"] = parts["keys"].copy()
    rng = np.random.default_rng(7 + m)
    c1 = parts["centers"][1]
    pick = rng.integers(0, c1.shape[1], size=(2, m))
    pick[:, ::5] = 0                                     # many keys as near to node 0 as to node 1
    new = np.stack([c1[t, pick[t]] + 0.3 * rng.normal(size=(m, d)) for t in range(2)]).astype(np.float32)
    new[:, ::10] = c1[:, :1]                             # and some on the two centres
    N = torch.from_numpy(new)[None].to(dtype).cuda()
    a, b = (HIPIndexer.from_layout(layout=layout, num_keys=int(held.min()), **parts) for _ in range(2))
    a.graft_min = b.graft_min = 1 << 30
    a.update(N, N)
    for i in range(m):
        b.update(N[:, :, i:i + 1], N[:, :, i:i + 1])
    assert a.size == b.size
    n = a.size[0]
    assert torch.equal(a.perm[:, :n], b.perm[:, :n])
    assert torch.equal(a.keys_buf[:, :n // 16 * 16], b.keys_buf[:, :n // 16 * 16])
    assert torch.equal(a.values_buf[:, :n], b.values_buf[:, :n])
    for l in (1, 2):
        k = a.size[l]
        assert torch.equal(a.counts[l][:, :k], b.counts[l][:, :k])
        assert torch.equal(a.radii[l][:, :k], b.radii[l][:, :k])
        assert torch.equal(a.centers_rowmajor(l)[:, :k], b.centers_rowmajor(l)[:, :k])
    if layout == "q8":
        assert torch.equal(a.keys8[:, :n], b.keys8[:, :n])  # (the capacities may differ)
        assert torch.equal(a.keps[:, :a.size[1]], b.keps[:, :b.size[1]])
    # the next window finds its nodes again
    a.update(N[:, :, :6], N[:, :, :6])
    for i in range(6):
        b.update(N[:, :, i:i + 1], N[:, :, i:i + 1])
    assert torch.equal(a.perm[:, :a.size[0]], b.perm[:, :b.size[0]])


@pytest.mark.parametrize("k2,bf,m,d,dtype,layout,bad", [
    (1, 8, 30, 64, torch.float32, "row_major", {5: "nan", 11: "inf", 12: "huge"}),
    (3, 8, 64, 128, torch.bfloat16, "row_major", {0: "huge", 63: "nan"}),            # first and last of a chunk
    (2, 16, 130, 128, torch.bfloat16, "tiled", {64: "inf", 65: "nan", 128: "huge"}),  # at the seams of chunks
    (3, 16, 80, 64, torch.bfloat16, "tiled", {3: "nan", 9: "inf"}),  # then more nodes with room than the list holds
    (1, 16, 40, 128, torch.bfloat16, "q8", {7: "huge"}),
])
def test_window_with_keys_that_have_no_distance(k2, bf, m, d, dtype, layout, bad, gpu_device):
    """A key whose distances are not finite opens a node of its own; the nodes with room stay known:
    the keys behind it, and the next windows, fill them as key by key."""
    from hira_amd.indexer.hip import HIPIndexer

    parts, held = _half_full(1, k2, bf, d, dtype, seed=m)
    rng = np.random.default_rng(m)
    c1 = parts["centers"][1]
    new = (c1[:, rng.integers(0, c1.shape[1], size=m)] + 0.3 * rng.normal(size=(1, m, d))).astype(np.float32)
    for i, what in bad.items():
        new[0, i, 3] = {"nan": np.nan, "inf": np.inf, "huge": 1e30}[what]  # (huge: its square overflows)
    N = torch.from_numpy(new)[None].to(dtype).cuda()
    a, b = (HIPIndexer.from_layout(layout=layout, num_keys=int(held[0]), **parts) for _ in range(2))
    for x in (a, b):
        x.graft_min = 1 << 30
        x.reserve(64 * bf * bf)  # (every such key may take a node of each level)
    free = int((bf - a.counts[1][:, :k2 * bf]).sum())
    bits = {torch.float32: torch.int32, torch.bfloat16: torch.int16}[dtype]

    def same():
        assert a.size == b.size and torch.equal(a._state[:, 1:], b._state[:, 1:])
        n = a.size[0]
        assert torch.equal(a.perm[:, :n], b.perm[:, :n])
        assert torch.equal(a.keys_buf.view(bits), b.keys_buf.view(bits))
        assert torch.equal(a.values_buf.view(bits)[:, :n], b.values_buf.view(bits)[:, :n])
        for l in (1, 2):
            k = a.size[l]
            assert torch.equal(a.counts[l][:, :k], b.counts[l][:, :k])
            assert torch.equal(a.radii[l][:, :k], b.radii[l][:, :k])
            assert torch.equal(a.centers_rowmajor(l).view(bits), b.centers_rowmajor(l).view(bits))

    a.update(N, N)
    for i in range(m):
        b.update(N[:, :, i:i + 1], N[:, :, i:i + 1])
    same()
    good = [i for i in range(m) if i not in bad]
    if len(good) <= free:  # the nodes that had room took them all
        assert int((bf - a.counts[1][:, :k2 * bf]).sum()) == free - len(good)
    for lo in (0, 6):  # the next windows find what room is left
        w = N[:, :, good[lo:lo + 6]].contiguous()
        a.update(w, w)
        for i in range(6):
            b.update(w[:, :, i:i + 1], w[:, :, i:i + 1])
        same()


@pytest.mark.parametrize("d,dv,dtype", [(260, 260, torch.float32), (264, 264, torch.bfloat16),
                                        (288, 288, torch.bfloat16), (312, 0, torch.bfloat16),
                                        (320, 320, torch.bfloat16), (320, 64, torch.bfloat16),
                                        (328, 328, torch.bfloat16)])
def test_windows_of_rows_beyond_256_columns(d, dv, dtype, gpu_device):
    """Around the widest rows that the list of nodes and a chunk of keys have room for."""
    from hira_amd.indexer.hip import HIPIndexer

    parts, held = _half_full(1, 2, 8, d, dtype, seed=d)
    parts["values"] = parts["keys"][:, :, :dv].copy() if dv <= d and dv else None
    rng = np.random.default_rng(d)
    m = 70
    c1 = parts["centers"][1]
    new = (c1[:, rng.integers(0, c1.shape[1], size=m)] + 0.3 * rng.normal(size=(1, m, d))).astype(np.float32)
    N = torch.from_numpy(new)[None].to(dtype).cuda()
    V = N[..., :dv].contiguous() if dv else None
    a, b = (HIPIndexer.from_layout(layout="row_major", num_keys=int(held[0]), **parts) for _ in range(2))
    a.graft_min = b.graft_min = 1 << 30
    a.update(N, V)
    for i in range(m):
        b.update(N[:, :, i:i + 1], None if V is None else V[:, :, i:i + 1])
    assert a.size == b.size
    n = a.size[0]
    assert torch.equal(a.perm[:, :n], b.perm[:, :n]) and torch.equal(a.keys_buf[:, :n], b.keys_buf[:, :n])
    if V is not None:
        assert torch.equal(a.values_buf[:, :n], b.values_buf[:, :n])
    for l in (1, 2):
        k = a.size[l]
        assert torch.equal(a.counts[l][:, :k], b.counts[l][:, :k])
        assert torch.equal(a.radii[l][:, :k], b.radii[l][:, :k])
        assert torch.equal(a.centers[l][:, :k], b.centers[l][:, :k])
