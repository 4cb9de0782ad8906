"""What HIPSearcher keeps between calls: no wait where an index has grown, launch options and outputs as
they are at the time of the call."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _index(n=3000, d=64, dtype=torch.float32, trees=2, seed=0, **kw):
    from hira_amd.indexer import HIPIndexer

    g = torch.Generator(device="cuda").manual_seed(seed)
    k, v = (torch.randn((1, trees, n, d), generator=g, device="cuda").to(dtype) for _ in range(2))
    return HIPIndexer(3, 1, 8, **kw).build(k, v), g


def test_a_search_without_a_scale_does_not_wait(gpu_device):
    from hira_amd.searcher import HIPSearcher

    idx, g = _index()
    idx.reserve(100)
    q, tau = torch.randn((4, 64), generator=g, device="cuda"), torch.full((4,), 8.0, device="cuda")
    new = torch.randn((1, 2, 1, 64), generator=g, device="cuda")
    se = HIPSearcher()
    for call in (lambda: se.search(q, tau, idx), lambda: se.search_attention(q, tau, idx)):
        call()
        idx.update(new, new, sync=False)
        call()  # (code and memory of a first call)
        torch.cuda.synchronize()
        size = list(idx.size)
        while idx.size == size:  # appends until the level sizes, and with them the call, are others
            idx.update(new, new, sync=False)
        torch.cuda.synchronize()
        torch.cuda._sleep(1_000_000_000)
        slept = torch.cuda.Event()
        slept.record()
        got = call()
        assert not slept.query(), "the host waited for what was enqueued before the search"
        torch.cuda.synchronize()
        want = HIPSearcher()
        ones = torch.ones((4,), device="cuda")
        ref = want.search(q, tau, idx, scaling=ones) if got.shape[1] == idx.size[0] else \
            want.search_attention(q, tau, idx, scaling=ones)
        assert torch.equal(got, ref) and bool((got != 0).any())


@pytest.mark.parametrize("trees,group", [(2, 4), (512, 8), (512, 9)])  # 8, 4096 and 4608 heads
def test_a_missing_scale_is_one(trees, group, gpu_device):
    from hira_amd.searcher import HIPSearcher

    idx, g = _index(n=40, trees=trees)
    h = trees * group
    q, tau = torch.randn((h, 64), generator=g, device="cuda"), torch.full((h,), 3.0, device="cuda")
    ones = torch.ones((h,), device="cuda")
    for _ in range(2):
        a = HIPSearcher()
        assert torch.equal(a.search(q, tau, idx).clone(), HIPSearcher().search(q, tau, idx, scaling=ones))
        assert torch.equal(a.search_attention(q, tau, idx), a.search_attention(q, tau, idx, scaling=ones))


def test_launch_options_are_those_of_the_call(gpu_device):
    from hira_amd import _lib
    from hira_amd.searcher import HIPSearcher

    idx, g = _index(n=9000, layout="row_major")
    q, tau = torch.randn((8, 64), generator=g, device="cuda"), torch.full((8,), 12.0, device="cuda")
    sc = torch.full((8,), 0.125, device="cuda")
    se = HIPSearcher(nodes_per_wave=200)
    ref = se.search_attention(q, tau, idx, scaling=sc).clone()
    dense = se.search(q, tau, idx, scaling=sc).clone()
    se.launch.nodes_per_wave = 1  # many more partials: a larger workspace
    assert torch.allclose(se.search_attention(q, tau, idx, scaling=sc), ref, rtol=1e-4, atol=1e-5)
    se.launch = _lib.HiraLaunch(64, 1, 1, 1)  # the same, folded by a second launch
    st = torch.zeros((2, _lib.HIRA_STATS_COLS), dtype=torch.int64, device="cuda")
    assert torch.allclose(se.search_attention(q, tau, idx, scaling=sc, stats=st), ref, rtol=1e-4, atol=1e-5)
    assert torch.equal(se.search(q, tau, idx, scaling=sc), dense)
    se.launch.kernel = 3
    for call in (se.search, se.search_attention):
        with pytest.raises(ValueError, match="kernel"):
            call(q, tau, idx, scaling=sc)
    se.launch = _lib.HiraLaunch(0, 0, 0, 0)
    assert torch.allclose(se.search_attention(q, tau, idx, scaling=sc), ref, rtol=1e-4, atol=1e-5)


def test_one_searcher_serves_indexes_of_any_number_of_trees(gpu_device):
    """The arrival counters of many trees lie where the partials of few did not write."""
    from hira_amd.searcher import HIPSearcher

    few, g = _index(n=9000, trees=2)
    many = [_index(n=n, trees=t, seed=t)[0] for t, n in ((300, 200), (96, 700), (9000, 40))]  # (18000 counters)
    se = HIPSearcher()
    for kernel in (0, 1):
        for idx in [few, many[0], few, many[1], many[2], many[0]]:
            h = idx.num_trees * 9
            q, tau = torch.randn((h, 64), generator=g, device="cuda"), torch.full((h,), 6.0, device="cuda")
            sc = torch.full((h,), 0.125, device="cuda")
            se.launch.kernel = kernel
            out = torch.full((h, 64), 7.0, device="cuda")
            se.search_attention(q, tau, idx, scaling=sc, out=out)
            assert torch.equal(out, HIPSearcher(kernel=kernel).search_attention(q, tau, idx, scaling=sc))


@pytest.mark.parametrize("layout", ["row_major", "tiled"])
def test_output_of_the_callers_own(layout, gpu_device):
    from hira_amd.indexer import HIPIndexer
    from hira_amd.searcher import HIPSearcher

    g = torch.Generator(device="cuda").manual_seed(1)
    k = torch.randn((1, 2, 3000, 64), generator=g, device="cuda").to(torch.bfloat16)
    idx = HIPIndexer(3, 1, 16, layout=layout).build(k, k)
    q, tau = torch.randn((8, 64), generator=g, device="cuda").to(torch.bfloat16), torch.full((8,), 12.0, device="cuda")
    sc = torch.full((8,), 0.125, device="cuda")
    se = HIPSearcher()
    ref = se.search_attention(q, tau, idx, scaling=sc)
    out = torch.full((2, 8, 64), 7.0, dtype=torch.bfloat16, device="cuda")  # (twice as much as is written)
    assert se.search_attention(q, tau, idx, scaling=sc, out=out) is out
    assert torch.equal(out[0], ref.to(torch.bfloat16)) and bool((out[1] == 7.0).all())
    assert torch.equal(se.search_attention(q, tau, idx, scaling=sc), ref)  # (fp32 again)
    assert torch.equal(se.search_attention(q, tau, idx, scaling=sc, out=torch.empty_like(ref)), ref)
    lists = se.search_compact(q, tau, idx)
    plan = se.plan_attention(idx, 8, scaling=sc)
    for bad in (torch.empty((8, 64), dtype=torch.float16, device="cuda"), torch.empty((8, 64)),
                torch.empty((8, 63), device="cuda"), torch.empty((64, 8), device="cuda").t()):
        with pytest.raises(ValueError):
            se.search_attention(q, tau, idx, scaling=sc, out=bad)
        with pytest.raises(ValueError):
            se.sparse_attention(*lists, idx, scaling=sc, out=bad)
    with pytest.raises(ValueError):
        se.sparse_attention(*lists, idx, scaling=sc, out=out)
    with pytest.raises(ValueError):
        plan.run(q, tau, torch.empty((8, 64), dtype=torch.float16, device="cuda"))
