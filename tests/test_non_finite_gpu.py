"""Values and scores that are not finite, on the vector-ALU search kernel: they reach the heads that
selected them and no other, and they reach those as a softmax over the selected keys in float64 has it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _expected(s, on, v, group):
    """Per head, over the selected rows alone (a row that is not selected is not multiplied by zero)."""
    out = torch.zeros((s.shape[0], v.shape[-1]), dtype=torch.float64)
    for h in range(s.shape[0]):
        rows = on[h].nonzero().squeeze(1)
        if len(rows):
            w = torch.softmax(s[h, rows], dim=0)
            out[h] = (w[:, None] * v[h // group, rows]).sum(0)
    return out


def _same(got, ref):
    got = got.double().cpu()
    assert torch.equal(got.isnan(), ref.isnan())
    assert torch.equal(got.isinf(), ref.isinf()) and torch.equal(got[got.isinf()], ref[ref.isinf()])
    fin = ref.isfinite()
    # (fp32 sums of fp32 / bf16 products against float64: as in the tests of finite values)
    assert float((got - ref)[fin].abs().max()) < 1e-4 * float(ref[fin].abs().max()) + 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("group", [1, 3, 8, 11])
@pytest.mark.parametrize("separate", [False, True])
def test_values_reach_only_the_heads_that_selected_them(dtype, group, separate, gpu_device):
    from hira_amd.indexer import HIPIndexer
    from hira_amd.searcher import HIPSearcher

    trees, n, d, m = 2, 5000, 64, 9
    g = torch.Generator().manual_seed(group)
    k, v = (torch.randn((1, trees, n, d), generator=g).to(dtype) for _ in range(2))
    q = torch.randn((trees * group, d), generator=g).to(dtype)
    qk, qv = (torch.randn((trees, m, d), generator=g).to(dtype) for _ in range(2))
    s = (k[0].double() @ q.double().reshape(trees, group, d).transpose(1, 2).contiguous()).transpose(1, 2)
    s = s.reshape(trees * group, n)
    top = s.topk(41, dim=1)
    tau = (0.5 * (top.values[:, 39] + top.values[:, 40])).float()
    on = s >= tau.double()[:, None]
    # of every third head: the key it likes best among those no other head of its tree selects
    by_tree = on.reshape(trees, group, n)
    for h in range(0, trees * group, 3):
        t = h // group
        alone = on[h] & (by_tree[t].sum(0) == 1)
        row = int(s[h].masked_fill(~alone, float("-inf")).argmax())
        v[0, t, row, h % 5] = float("inf")
        v[0, t, row, 7 + h % 5] = float("-inf")
        v[0, t, row, 20 + h % 5] = float("nan")
    idx = HIPIndexer(3, 1, 8, layout="row_major").build(k.cuda(), v.cuda())
    se = HIPSearcher(kernel=1, separate_merge=separate)
    sc = torch.full((trees * group,), d ** -0.5, device="cuda")
    ref = _expected(s * d ** -0.5, on, v[0].double(), group)
    assert ref.isinf().any() and ref.isnan().any() and ref.isfinite().all(1).any()
    _same(se.search_attention(q.cuda(), tau, idx, scaling=sc), ref)
    # the same with a queue, whose keys every head takes: one of its values is not finite in tree 1
    qv[1, 4, 60] = float("inf")
    sq = (qk.double() @ q.double().reshape(trees, group, d).transpose(1, 2).contiguous()).transpose(1, 2)
    s2 = torch.cat([s, sq.reshape(trees * group, m)], 1) * d ** -0.5
    on2 = torch.cat([on, torch.ones((trees * group, m), dtype=torch.bool)], 1)
    ref = _expected(s2, on2, torch.cat([v[0], qv], 1).double(), group)
    _same(se.search_attention(q.cuda(), tau, idx, scaling=sc, queue_keys=qk.cuda(), queue_values=qv.cuda()), ref)


@pytest.mark.parametrize("group", [1, 4, 5])
@pytest.mark.parametrize("separate", [False, True])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_scores_that_are_no_numbers_are_not_dropped(group, separate, bad, gpu_device):
    """A queued key is selected whatever it scores; a score that is NaN, or infinite, leaves no
    finite softmax."""
    from hira_amd.indexer import HIPIndexer
    from hira_amd.searcher import HIPSearcher

    trees, n, d, m = 2, 2000, 64, 5
    g = torch.Generator().manual_seed(3)
    k, v = (torch.randn((1, trees, n, d), generator=g).cuda() for _ in range(2))
    q = torch.randn((trees * group, d), generator=g).abs()  # (an infinite column: an infinite score)
    qk, qv = (torch.randn((trees, m, d), generator=g) for _ in range(2))
    qk[1, 2, 10] = bad
    idx = HIPIndexer(3, 1, 8, layout="row_major").build(k, v)
    se = HIPSearcher(kernel=1, separate_merge=separate)
    for tau in (20.0, 1e30):  # some keys of the index, none
        out = se.search_attention(q.cuda(), tau, idx, queue_keys=qk.cuda(), queue_values=qv.cuda())
        assert bool(out[:group].isfinite().all()) and bool(out[group:].isnan().all())
