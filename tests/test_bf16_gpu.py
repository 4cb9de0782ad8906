"""fp32 numbers become bf16 by an instruction: to the nearest, ties to even, a NaN stays one.  Against torch's conversion on
the CPU, bit for bit, through the attention output of one key a tree and through the centres of blocks of two keys."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bits(x):
    return x.view(torch.int16).to(torch.int32) & 0xffff


@pytest.mark.parametrize("low", [0x0000, 0x0001, 0x7fff, 0x8000, 0x8001, 0xffff])
def test_every_number_of_the_upper_half_is_rounded(low, gpu_device):
    """All 65536 upper halves of a word over lower halves at, below and above a tie: zeros, subnormal numbers, infinities and
    NaN of any payload among them."""
    from hira_amd.indexer import HIPIndexer
    from hira_amd.searcher import HIPSearcher

    h, d = 256, 256
    words = torch.arange(65536, dtype=torch.int64) << 16 | low
    vals = (words - ((words >> 31) << 32)).to(torch.int32).view(torch.float32).reshape(1, h, 1, d)
    keys = torch.ones((1, h, 1, 64))
    idx = HIPIndexer(2, 1, 16).build(keys.cuda(), vals.cuda())
    plan = HIPSearcher().plan_attention(idx, h, scaling=torch.ones(h))
    out = torch.empty((h, d), dtype=torch.bfloat16, device="cuda")
    plan.run(torch.ones((h, 64), device="cuda"), torch.full((h,), -3e38, device="cuda"), out)  # 0 + 1 * value
    want, got = vals.reshape(h, d).to(torch.bfloat16), out.cpu()
    nan = vals.reshape(h, d).isnan()
    assert nan.any() and torch.equal(got.isnan(), nan)
    same = (_bits(got) == _bits(want)) | nan | ((got == 0) & (want == 0))
    assert same.all(), [hex(int(w)) for w in words.reshape(h, d)[~same][:8]]


@pytest.mark.parametrize("n", [600, 9000])
@pytest.mark.parametrize("d", [64, 128])
def test_block_centres_are_rounded(n, d, gpu_device):
    """The mean of two bf16 numbers is exact in fp32 but for far exponents, and half of those whose exponents differ by one
    are ties: levels that one launch takes whole, and larger ones."""
    from hira_amd.indexer import HIPIndexer

    g = torch.Generator().manual_seed(n + d)
    keys = (torch.randn((1, 2, n, d), generator=g) * 2.0 ** torch.randint(-5, 6, (1, 2, n, d), generator=g)).to(torch.bfloat16)
    idx = HIPIndexer(2, 1, 2).build(keys.cuda(), keys.cuda())
    k = idx.size[1]
    a, b = (idx.keys_rowmajor()[:, i:2 * k:2].float().cpu() for i in (0, 1))
    whole = (idx.counts[1][:, :k] == 2).cpu()
    want, got = ((a + b) / 2).to(torch.bfloat16), idx.centers[1][:, :k].cpu()
    ties = (_bits((a + b)[whole].view(torch.int32).view(torch.int16).reshape(-1, 2)[:, 0]) == 0x8000).sum()
    assert whole.sum() > n // 4 and ties > 100
    assert torch.equal(_bits(got[whole]), _bits(want[whole]))
