"""A subtree clustered anew by the library, against the same steps taken one by one: a two-level build of the
keys the subtree holds, its nodes moved to the front, the radii above from their definition."""

import numpy as np
import pytest
import torch

from helpers import bf16_round, clustered_keys

pytestmark = pytest.mark.gpu


def _rows(idx, l):
    """Level l of an index (0: keys) row by row."""
    from hira_amd.indexer.hip import from_tiled

    x = idx.keys_buf if l == 0 else idx.centers[l]
    return from_tiled(x) if (idx.keys_tiled if l == 0 else idx.tiled) else x


@pytest.mark.parametrize("dtype,d,bf,levels,layout,vals", [
    (torch.bfloat16, 128, 32, 3, "auto", True),    # 1024 rows: a workgroup a tree; an 8-bit shadow
    (torch.bfloat16, 256, 32, 3, "auto", True),    # launches
    (torch.bfloat16, 64, 16, 4, "tiled", False),
    (torch.bfloat16, 72, 8, 5, "auto", True),      # rows that do not fill their lanes
    (torch.float32, 32, 8, 4, "auto", True),
    (torch.float32, 4, 3, 4, "auto", True),
])
def test_a_subtree_is_clustered_as_an_index_of_its_keys(dtype, d, bf, levels, layout, vals, gpu_device):
    from hira_amd.indexer.hip import HIPIndexer

    t = 3
    n0 = 2 * bf * bf + bf + 1 if levels == 3 else bf ** 3 + 2 * bf * bf + 1
    m = bf * bf // 2 + 1
    rnd = bf16_round if dtype == torch.bfloat16 else (lambda x: x)
    keys = rnd(clustered_keys(t, n0 + m, d, seed=bf + d, clusters=9))
    K = torch.from_numpy(keys)[None].to(dtype)
    V = torch.from_numpy(rnd(np.random.default_rng(1).normal(size=(t, n0 + m, d)).astype(np.float32)))[None].to(dtype)
    idx = HIPIndexer(levels, 2, bf, layout=layout).build(K[:, :, :n0], V[:, :, :n0] if vals else None)
    idx.update(K[:, :, n0:], V[:, :, n0:] if vals else None)
    nsub = bf * bf
    for node in (0, idx.size[2] - 1):
        s0, b0 = node * nsub, node * bf
        perm = idx.perm[:, s0:s0 + nsub].clone()
        live = perm >= 0
        order = torch.sort((~live).to(torch.uint8), dim=1, stable=True).indices

        def front(x):
            return torch.gather(x[:, s0:s0 + nsub], 1, order[:, :, None].expand(-1, -1, x.shape[2]))

        sub = HIPIndexer(2, 2, bf, seed=idx.seed + node, pack_rounds=idx.pack_rounds, layout=idx.layout_name).build(
            front(_rows(idx, 0))[None], front(idx.values_buf)[None] if vals else None,
            key_counts=live.sum(dim=1, dtype=torch.int32))
        nodes = torch.sort((sub.counts[1][:, :bf] == 0).to(torch.uint8), dim=1, stable=True).indices
        slots = (nodes[:, :, None] * bf + torch.arange(bf, device=nodes.device)).reshape(t, nsub)
        pos = torch.gather(perm, 1, order)
        sp = torch.gather(sub.perm[:, :nsub], 1, slots).long()
        want_perm = torch.where(sp >= 0, torch.gather(pos, 1, sp.clamp(min=0)), -1)
        want = {l: _rows(idx, l).clone() for l in range(levels)}
        want[0][:, s0:s0 + nsub] = torch.gather(_rows(sub, 0)[:, :nsub], 1, slots[:, :, None].expand(-1, -1, d))
        want[1][:, b0:b0 + bf] = torch.gather(_rows(sub, 1)[:, :bf], 1, nodes[:, :, None].expand(-1, -1, d))
        radii, counts = [None if r is None else r.clone() for r in idx.radii], [None if c is None else c.clone() for c in idx.counts]
        radii[1][:, b0:b0 + bf] = torch.gather(sub.radii[1][:, :bf], 1, nodes)
        counts[1][:, b0:b0 + bf] = torch.gather(sub.counts[1][:, :bf], 1, nodes)
        counts[2][:, node] = (counts[1][:, b0:b0 + bf] > 0).sum(dim=1, dtype=torch.int32)
        child = node
        for l in range(2, levels):
            here = want[l][:, child].double()
            if l == 2:
                need = ((want[1][:, b0:b0 + bf].double() - here[:, None]).norm(dim=2) + radii[1][:, b0:b0 + bf].double()).amax(dim=1)
            else:
                below = want[l - 1][:, child * bf:child * bf + bf]
                at = last % bf
                need = (below[:, at].double() - here).norm(dim=1) + radii[l - 1][:, last].double()
                need = torch.maximum(need, radii[l][:, child].double())
            radii[l][:, child] = need.float()
            last, child = child, child // bf
        want_values = None
        if vals:
            want_values = idx.values_buf.clone()
            want_values[:, s0:s0 + nsub] = torch.gather(sub.values_buf[:, :nsub], 1, slots[:, :, None].expand(-1, -1, d))
        want_all = idx.perm.clone()
        want_all[:, s0:s0 + nsub] = want_perm

        idx.rebuild_subtree(node)
        assert torch.equal(idx.perm, want_all)
        if vals:
            assert torch.equal(idx.values_buf, want_values)
        for l in range(levels):
            assert torch.equal(_rows(idx, l), want[l]), l
        for l in range(1, levels):
            assert torch.equal(idx.counts[l], counts[l]), l
            if l == 1:
                assert torch.equal(idx.radii[1], radii[1])
                continue
            # the radius covers what it has to (but for the rounding of sums of d squares in fp32, each of
            # (d + 3) half units in the last place at most), and exceeds it by its head room of 1e-6 a level
            a, b = idx.radii[l].double(), radii[l].double()
            eps = (d + 3) * 2.0 ** -24
            ok = (a == b) | ((a >= b * (1 - eps)) & (a <= b * (1 + eps + 1e-6 * levels + 2.0 ** -22)))
            assert bool(ok.all()), (l, a[~ok], b[~ok])
        if idx._state is not None:
            assert int(idx._state[:, 0].abs().max()) == 0
        if idx.q8:
            again = idx.keys8.clone()
            idx.quantize(s0, nsub)
            assert torch.equal(again, idx.keys8)
