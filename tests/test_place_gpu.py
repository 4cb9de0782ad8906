"""Keys, values and centres in their slots, radii and counts: value rows of widths that take another way, indexes
of up to six levels, with empty slots and empty nodes, against the same by tensor operations."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,n,d,dv,levels,bf,layout", [
    (torch.bfloat16, 1000, 64, 64, 6, 4, "auto"),
    (torch.bfloat16, 1111, 64, 1024, 3, 10, "auto"),   # a value row is more than a wave's 16 bytes a lane
    (torch.bfloat16, 777, 128, 8, 3, 32, "auto"),
    (torch.bfloat16, 500, 40, 72, 2, 64, "auto"),
    (torch.float32, 333, 36, 260, 4, 3, "auto"),
    (torch.float32, 65, 256, 4, 1, 8, "auto"),
    (torch.bfloat16, 65, 64, 520, 1, 8, "auto"),
    (torch.bfloat16, 900, 128, 128, 3, 16, "q8"),      # a small first level
    (torch.bfloat16, 5000, 64, 64, 3, 16, "q8"),
])
def test_rows_radii_and_counts(dtype, n, d, dv, levels, bf, layout, gpu_device):
    from hira_amd.indexer.hip import HIPIndexer

    g = torch.Generator().manual_seed(n)
    keys = torch.randn(1, 2, n, d, generator=g).to(dtype).to(gpu_device)
    values = torch.randn(1, 2, n, dv, generator=g).to(dtype).to(gpu_device)
    index = HIPIndexer(levels, 1, bf, layout=layout).build(keys, values)
    torch.cuda.synchronize()
    size0 = index.size[0]
    for t in range(2):
        perm = index.perm[t, :size0].long()
        live = perm >= 0
        assert sorted(perm[live].tolist()) == list(range(n))
        for got, rows in ((index.keys_rowmajor()[t, :size0], keys[0, t]), (index.values_buf[t, :size0], values[0, t])):
            assert torch.equal(got, torch.where(live[:, None], rows[perm.clamp(min=0)], torch.zeros_like(rows[:1])))
        child, child_live, child_r = index.keys_rowmajor()[t, :size0].double(), live, torch.zeros(size0, device=gpu_device)
        for l in range(1, levels):
            m = index.size[l]
            c = index.centers_rowmajor(l)[t, :m].double()
            count = child_live.reshape(m, bf).sum(1)
            assert torch.equal(index.counts[l][t, :m].long(), count)
            r = index.radii[l][t, :m]
            assert bool((torch.isneginf(r) == (count == 0)).all())
            dist = (child.reshape(m, bf, d) - c[:, None]).norm(dim=-1) + child_r.double().reshape(m, bf)
            want = dist.masked_fill(~child_live.reshape(m, bf), float("-inf")).max(1).values
            ok = count > 0
            # fp32 sums of d squares, a root, and the few ulp of head room
            assert torch.allclose(r[ok].double(), want[ok], rtol=(d + 8) * 2 ** -24 * 2, atol=1e-6)
            assert bool((r[ok].double() >= want[ok] * (1 - 2e-7)).all())
            child, child_live, child_r = c, ok, torch.where(ok, r, torch.zeros_like(r))
    if layout == "q8":
        step = keys[0].float().abs().amax(1).cpu() / 127.0  # (on the CPU: a division, not a product)
        np.testing.assert_array_equal(index.kscale.cpu().numpy(), step.numpy())
