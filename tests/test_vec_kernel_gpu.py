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


@pytest.mark.parametrize("trees,n,d,levels,bf,group,queue", [
    (50, 1200, 32, 2, 4, 2, 1),     # 250 workgroups for the trees, or 200 and 50 for the queues
    (50, 1200, 32, 2, 4, 2, 130),   # three blocks of queued rows, one workgroup
    (8, 5003, 96, 4, 16, 3, 33),
    (130, 300, 16, 2, 4, 1, 64),    # no place to keep: more queues than half of the compute units
])
def test_a_place_for_every_queue(trees, n, d, levels, bf, group, queue, gpu_device):
    print(f"case trees={trees} n={n} d={d} queue={queue}", flush=True)
    _check(n, d, torch.bfloat16 if d == 96 else torch.float32, levels, bf, group, seed=n + queue, queue=queue, trees=trees)


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


ONE_CASES = [
    # trees, heads a tree, keys, key width, value width, fan-out, levels, type, layout, queued rows
    (1, 1, 9, 16, 16, 1, 3, torch.float32, "row_major", 0),      # fan-out 1: as many nodes as keys
    (2, 1, 500, 128, 64, 2, 5, torch.float32, "row_major", 0),   # more rows of level 2 than a load brings
    (2, 3, 777, 64, 128, 3, 7, torch.bfloat16, "row_major", 40),
    (1, 4, 2100, 80, 80, 7, 4, torch.float32, "row_major", 129),
    (3, 5, 600, 256, 256, 64, 2, torch.float32, "row_major", 3),   # a node is half a workgroup's rows
    (2, 8, 640, 512, 512, 16, 3, torch.bfloat16, "row_major", 0),  # 64 lanes a row, eight heads
    (2, 12, 1500, 96, 96, 10, 3, torch.bfloat16, "tiled", 9),
    (2, 4, 3000, 64, 64, 4, 2, torch.bfloat16, "tiled", 0),
    (1, 2, 1300, 8, 8, 5, 4, torch.bfloat16, "row_major", 1),
]


@pytest.mark.parametrize("t,g,n,d,dv,bf,nl,dtype,layout,m", ONE_CASES)
def test_one_block_a_wave_equals_the_general_way(t, g, n, d, dv, bf, nl, dtype, layout, m, gpu_device):
    """Launches whose workgroups ask for their keys beside the gates, against the batches and lists that
    launch options still take: the same scores, lists and counters, attention but for the order of its
    sums, also with heads in an order of the caller's, key and value rows that are not finite, a head
    that selects everything and one that selects nothing."""
    from hira_amd.indexer import HIPIndexer
    from hira_amd.searcher import HIPSearcher

    print(f"case {t} {g} {n} {d} {dv} {bf} {nl} {dtype} {layout} {m}", flush=True)
    gen = torch.Generator().manual_seed(n + d)
    k = torch.randn(1, t, n, d, generator=gen).to(dtype).cuda()
    v = torch.randn(1, t, n, dv, generator=gen).to(dtype).cuda()
    q = torch.randn(t * g, d, generator=gen).to(dtype).cuda()
    idx = HIPIndexer(nl, 1, bf, layout=layout).build(k, v)
    s = torch.matmul(q.reshape(t, g, d).float(), k[0].float().transpose(1, 2).contiguous()).reshape(t * g, n)
    tau = s.topk(max(1, n // 20), dim=1).values[:, -1].contiguous()
    tau[0] = float("inf") if t * g > 1 else tau[0]
    tau[-1] = float("-inf")
    qk = qv = None
    if m:
        qk, qv = (torch.randn(t, m, w, generator=gen).to(dtype).cuda() for w in (d, dv))
    sc = torch.full((t * g,), d ** -0.5, device="cuda")
    one, gen_way = HIPSearcher(kernel=1), HIPSearcher(kernel=1, nodes_per_wave=3)
    turned = torch.arange(t).repeat(g) if t > 1 else None
    for q2kv in (None, turned):
        out = []
        for se in (one, gen_way):
            st = torch.zeros((t, 11), dtype=torch.int64, device="cuda")
            dense = se.search(q, tau, idx, q_head_to_kv=q2kv, scaling=sc, stats=st).clone()
            pos = se.search(q, tau, idx, q_head_to_kv=q2kv, index_space="position").clone()
            at, score, count = (x.clone() for x in se.search_compact(q, tau, idx, q_head_to_kv=q2kv))
            by = torch.full((t * g, idx.size[0]), -9.0, device="cuda")
            for h in range(t * g):
                by[h, at[h, : count[h]].long()] = score[h, : count[h]]
            att = se.search_attention(q, tau, idx, q_head_to_kv=q2kv, scaling=sc, queue_keys=qk, queue_values=qv)
            out.append((dense, pos, by, count, st, att))
        for a, b in zip(out[0][:5], out[1][:5]):
            assert torch.equal(a, b)
        a, b = out[0][5], out[1][5]
        assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())  # (sums of fp32 in another order)
    slot = int((idx.perm[0] >= 0).nonzero()[0])
    idx.values_buf[0, slot] = float("inf")
    if not idx.tiled:
        idx.keys_buf[0, slot + (idx.perm[0, slot + 1] >= 0).int().item()] = float("nan")
    a, b = (se.search_attention(q, tau, idx, scaling=sc, queue_keys=qk, queue_values=qv) for se in (one, gen_way))
    assert torch.equal(a.isfinite(), b.isfinite()) and torch.equal(a.isnan(), b.isnan())


def _chain_of_fmas(x, q):
    """Scores (T, G, N) of bf16 rows x (T, N, D) and q (T, G, D) as a lane's chain of fmas over its chunk gives them (the
    products are exact in 32 bits) and the lanes' sums in the kernel's order."""
    t, n, d = x.shape
    lanes = 1
    while lanes * 8 < d:
        lanes *= 2
    c = torch.zeros(t, q.shape[1], n, lanes)
    for e in range(8):
        p = q[:, :, None, e::8].float() * x[:, None, :, e::8].float()
        c[..., :p.shape[-1]] += p
    while lanes > 1:
        lanes //= 2
        high = c[..., lanes:]
        c = c[..., :lanes] + (high if lanes >= 16 else high.flip(-1))
    return c[..., 0]


@pytest.mark.parametrize("large", [0, 8])
@pytest.mark.parametrize("d", [16, 32, 96, 128, 256])
def test_bf16_scores_are_no_further_from_64_bits(d, large, gpu_device):
    """Products two an instruction: the error against 64 bits is that of a chain of fmas."""
    from hira_amd.indexer import HIPIndexer
    from hira_amd.searcher import HIPSearcher

    t, g, n = 2, 8, 3000
    gen = torch.Generator().manual_seed(d + large)
    x, q = torch.randn(t, n, d, generator=gen), torch.randn(t, g, d, generator=gen)
    x[..., :large] *= 20.0
    x, q = x.bfloat16(), q.bfloat16()
    index = HIPIndexer(2, 0, 16, layout="row_major").build(x[None].cuda())
    got = HIPSearcher(kernel=1, index_space="position").search(q.reshape(t * g, d).cuda(), float("-inf"), index)
    want = torch.matmul(q.double(), x.double().transpose(1, 2).contiguous())
    err = got.cpu().double().reshape(t, g, n) - want
    # (two roundings in each of two instructions, the halves, the lanes, each at most 2^-23 of the sum of magnitudes)
    most = torch.matmul(q.double().abs(), x.double().abs().transpose(1, 2).contiguous())
    assert float((err.abs() / most).max()) <= (5 + max(0, d // 8 - 1).bit_length()) * 2.0 ** -23
    chain = _chain_of_fmas(x, q).double() - want
    # 48000 scores: the two root mean squares vary by a hundredth
    assert float(err.square().mean().sqrt()) <= 1.05 * float(chain.square().mean().sqrt())


@pytest.mark.parametrize("exponent", [0, 100])
@pytest.mark.parametrize("d", [16, 96, 256])
def test_bf16_rows_of_subnormal_numbers(d, exponent, gpu_device):
    """Rows below the normal range count in full: whole multiples of 2^-133, whose sums are exact."""
    from hira_amd.indexer import HIPIndexer
    from hira_amd.searcher import HIPSearcher

    gen = torch.Generator().manual_seed(d)
    k = torch.randint(-127, 128, (2, 500, d), generator=gen)
    x = torch.where(k < 0, -k - 2 ** 15, k).to(torch.int16).view(torch.bfloat16)  # (the bits: a sign and a multiple)
    assert torch.equal(x.double(), k.double() * 2.0 ** -133)
    whole = torch.randint(-9, 10, (2, 3, d), generator=gen)
    q = (whole.double() * 2.0 ** exponent).bfloat16()
    index = HIPIndexer(1, 0, 16, layout="row_major").build(x[None].cuda())
    got = HIPSearcher(kernel=1, index_space="position").search(q.reshape(6, d).cuda(), float("-inf"), index)
    want = torch.matmul(whole.double(), k.double().transpose(1, 2).contiguous()) * 2.0 ** (exponent - 133)
    assert torch.equal(got.cpu().double().reshape(2, 3, 500), want)
