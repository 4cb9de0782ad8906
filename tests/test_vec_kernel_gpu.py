"""The vector-ALU search kernel where its shapes can go wrong: every number of lanes a row takes, head
groups around the passes of 1 / 4 / 8, fan-outs 1, 2 and 64, deep trees, node counts around a batch
of 64, small workgroups; against brute force in float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(n, d, dtype, levels, bf, group, seed, queue=0, trees=2, **kw):
    from hira_amd.indexer import HIPIndexer
    from hira_amd.searcher import HIPSearcher

    g = torch.Generator().manual_seed(seed)
    k, v = (torch.randn((1, trees, n, d), generator=g).to(dtype).cuda() for _ in range(2))
    q = torch.randn((trees * group, d), generator=g).to(dtype).cuda()
    s = torch.einsum("tnd,tgd->tgn", k[0].double(), q.double().reshape(trees, group, d)).reshape(trees * group, n)
    keep = max(1, n // 7)
    top = s.topk(min(keep + 1, n), dim=1).values
    tau = (0.5 * (top[:, keep - 1] + top[:, -1])).float() if n > keep else top[:, -1].float() - 1e-3
    idx = HIPIndexer(levels, 1, bf, layout="row_major").build(k, v)
    se = HIPSearcher(kernel=1, index_space="position", **kw)
    want = torch.where(s >= tau.double()[:, None], s, torch.zeros_like(s))
    got = se.search(q, tau, idx).double()
    assert torch.equal(got != 0, want != 0)
    assert torch.allclose(got, want, rtol=2e-5, atol=1e-5)
    slots = HIPSearcher(kernel=1, output_fill_value=-7.0, **kw).search(q, tau, idx)  # the fused fill
    assert int((slots != -7.0).sum()) == int((want != 0).sum())
    lists = se.search_compact(q, tau, idx)
    assert torch.equal(lists[2].long(), (want != 0).sum(1))
    qk = qv = None
    vq = v[0].double().repeat_interleave(group, 0)
    z, on = s * d ** -0.5, want != 0
    if queue:
        qk, qv = (torch.randn((trees, queue, d), generator=g).to(dtype).cuda() for _ in range(2))
        sq = torch.einsum("tnd,tgd->tgn", qk.double(), q.double().reshape(trees, group, d)).reshape(trees * group, queue)
        z, on = torch.cat([z, sq * d ** -0.5], 1), torch.cat([on, torch.ones_like(sq, dtype=torch.bool)], 1)
        vq = torch.cat([vq, qv.double().repeat_interleave(group, 0)], 1)
    w = torch.softmax(z.masked_fill(~on, float("-inf")), dim=1)
    ref = torch.einsum("hn,hnd->hd", w, vq)
    out = se.search_attention(q, tau, idx, scaling=torch.full((trees * group,), d ** -0.5, device="cuda"),
                              queue_keys=qk, queue_values=qv)
    assert float((out.double() - ref).abs().max()) < 1e-4 * float(ref.abs().max()) + 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d", [8, 16, 32, 40, 64, 80, 128, 200, 256])
@pytest.mark.parametrize("group", [1, 3, 8])
def test_row_widths_and_head_groups(dtype, d, group, gpu_device):
    _check(517, d, dtype, 3, 6, group, seed=d + group, queue=5)


@pytest.mark.parametrize("n,levels,bf,group", [(1, 2, 4, 1), (63 * 4, 2, 4, 4), (64 * 4, 2, 4, 4), (65 * 4 + 1, 2, 4, 5),
                                               (300, 4, 1, 2), (700, 8, 2, 4), (3000, 6, 3, 9), (4100, 2, 64, 4),
                                               (900, 1, 8, 3), (12001, 3, 64, 17)])
def test_trees_and_batches(n, levels, bf, group, gpu_device):
    _check(n, 64, torch.float32, levels, bf, group, seed=n, queue=70)


@pytest.mark.parametrize("threads,npw", [(64, 1), (64, 70), (128, 3), (256, 33), (512, 9)])
def test_workgroup_shapes(threads, npw, gpu_device):
    _check(2500, 80, torch.float32, 3, 7, 4, seed=threads + npw, queue=33, block_threads=threads, nodes_per_wave=npw)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_first_call_on_an_index_may_be_captured(dtype, gpu_device):
    """No scale given, another index than the call before (same heads): nothing comes from the host."""
    from hira_amd.indexer import HIPIndexer
    from hira_amd.searcher import HIPSearcher

    keys, vals = (torch.randn(2, 1, 2, 900, 64, device="cuda").to(dtype) for _ in range(2))
    a, b = (HIPIndexer(2, 1, 32).build(k, v) for k, v in zip(keys, vals))
    q, tau = torch.randn(4, 64, device="cuda").to(dtype), torch.full((4,), 6.0, device="cuda")
    searcher = HIPSearcher()
    searcher.search_attention(q, tau, a)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = searcher.search_attention(q, tau, b)
    want = HIPSearcher().search_attention(q, tau, b, scaling=torch.ones(4, device="cuda"))
    assert bool((want != 0).any())
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
