"""The 8-bit shadow against the division it stands for, taken on the host: steps of any mantissa, keys of all sizes,
infinities and NaN."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,bf,spread", [(128, 32, 1), (64, 16, 1), (128, 16, 40)])
def test_shadow_is_the_rounded_quotient(d, bf, spread, gpu_device):
    from hira_amd.indexer.hip import HIPIndexer, from_tiled

    t, n = 2, 40 * bf + 3
    rng = np.random.default_rng(d + bf + spread)
    keys = rng.normal(size=(1, t, n, d)) * np.exp(rng.normal(size=(1, t, n, d)) * np.log(spread) if spread > 1 else 0.0)
    keys[0, 0, 5, 3], keys[0, 0, 9, 4], keys[0, 1, 7, :] = np.inf, np.nan, 0.0
    K = torch.from_numpy(keys.astype(np.float32)).to(torch.bfloat16).cuda()
    idx = HIPIndexer(2, 1, bf, layout="q8").build(K, K)
    rows = idx.keys_buf if not idx.keys_tiled else from_tiled(idx.keys_buf)
    for new_steps in (False, True):
        if new_steps:
            step = np.exp2(rng.uniform(-12, 3, size=(t, d))).astype(np.float32)  # (some clip, some underflow)
            idx.kscale.copy_(torch.from_numpy(step).reshape(idx.kscale.shape))
            idx.quantize(0, idx.size[0])
        step = idx.kscale.cpu().numpy().reshape(t, 1, d)
        m = idx.size[0]
        f, live = rows[:, :m].float().cpu().numpy(), (idx.perm[:, :m] >= 0).cpu().numpy()
        with np.errstate(all="ignore"):
            v = (f / step).astype(np.float32)
            r = np.fmin(np.fmax(np.rint(v), np.float32(-127)), np.float32(127))
            err = np.abs(v - r)
        r, err = np.where(live[:, :, None], r, 0), np.where(live[:, :, None], err, 0)
        s, j = np.arange(m)[:, None], np.arange(d)[None]
        at = (((s // 16) * (d // 64) + j // 64) * 64 + ((j % 64) // 16) * 16 + s % 16) * 16 + j % 16
        got = idx.keys8.reshape(t, -1).cpu().numpy()[:, at]
        assert np.array_equal(got, r.astype(np.int8))
        worst = np.fmax.reduce(np.fmax(err, 0).reshape(t, m // bf, bf * d), axis=2).astype(np.float32)
        assert np.array_equal(idx.keps[:, :m // bf].cpu().numpy(), worst)
