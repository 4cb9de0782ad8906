"""hira_enqueue, hira_replace_rows and hira_fill_arrays against the same moves in torch, and the
bf16 attention output against the rounded fp32 one."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("trees,cap,at,m,d,dv", [(1, 1, 0, 1, 8, 8), (3, 7, 2, 5, 80, 24), (128, 16, 15, 1, 128, 128),
                                                 (2, 300, 0, 300, 256, 8)])
def test_enqueue(dtype, trees, cap, at, m, d, dv, gpu_device):
    from hira_amd import _lib

    qk, qv = torch.randn(trees, cap, d, device="cuda").to(dtype), torch.randn(trees, cap, dv, device="cuda").to(dtype)
    k, v = torch.randn(trees, m, d, device="cuda").to(dtype), torch.randn(trees, m, dv, device="cuda").to(dtype)
    wk, wv = qk.clone(), qv.clone()
    wk[:, at:at + m], wv[:, at:at + m] = k, v
    code = _lib.HIRA_F32 if dtype == torch.float32 else _lib.HIRA_BF16
    _lib.check(_lib.lib().hira_enqueue(qk.data_ptr(), qv.data_ptr(), code, trees, cap, at, m, d, dv, k.data_ptr(),
                                       v.data_ptr(), _lib.current_stream(qk.device)))
    assert torch.equal(qk, wk) and torch.equal(qv, wv)
    with pytest.raises(ValueError):
        _lib.check(_lib.lib().hira_enqueue(qk.data_ptr(), qv.data_ptr(), code, trees, cap, cap, m, d, dv, k.data_ptr(),
                                           v.data_ptr(), _lib.current_stream(qk.device)))


@pytest.mark.parametrize("n", [1, 32, 33, 130, 300, 448, 449, 900])
def test_replace_rows(n, gpu_device):
    from hira_amd import _lib

    trees, rows, d, m, stride = 3, 1000, 72, 310, 320
    a = torch.randn(trees, rows, d, device="cuda").to(torch.bfloat16)
    src = torch.randn(trees, stride, d, device="cuda").to(torch.bfloat16)
    slot, frm = torch.randperm(rows)[:n], torch.randint(0, m, (n,))
    want = a.clone()
    want[:, slot.cuda()] = src[:, frm.cuda()]
    arr = C.c_int32 * n
    args = (a.data_ptr(), _lib.HIRA_BF16, d, trees, rows, src.data_ptr(), m, stride, arr(*slot.tolist()),
            arr(*frm.tolist()))
    _lib.check(_lib.lib().hira_replace_rows(*args, n, _lib.current_stream(a.device)))
    assert torch.equal(a, want)
    bad = args[:-2] + (arr(*([rows] * n)), args[-1])
    with pytest.raises(ValueError):
        _lib.check(_lib.lib().hira_replace_rows(*bad, n, _lib.current_stream(a.device)))


@pytest.mark.parametrize("trees", [1, 5])
def test_fill_arrays(trees, gpu_device):
    from hira_amd.indexer.hip import _fill_arrays

    specs, wants = [], []
    # (rows, width, rows of the source, rows copied, first row filled): whole stretches and ragged ones,
    # 16-byte rows and single words, a gap that stays as it is
    for rows, width, have, copied, first in [(5000, 64, 4000, 4000, 4000), (7, 0, 3, 3, 3), (40000, 0, 0, 0, 11),
                                             (33, 8, 40, 20, 25), (1, 4, 0, 0, 0), (9000, 0, 9000, 9000, 9000)]:
        shape = (trees, rows) + ((width,) if width else ())
        dst = torch.randn(shape, device="cuda")
        src = torch.randn((trees, have) + shape[2:], device="cuda") if have else None
        want = dst.clone()
        if copied:
            want[:, :copied] = src[:, :copied]
        want[:, first:] = float("-inf")
        specs.append((dst, src, copied, first, 0xFF800000))
        wants.append(want)
    _fill_arrays(specs, trees)
    for (dst, *_), want in zip(specs, wants):
        assert torch.equal(dst, want)


@pytest.mark.parametrize("dtype,d,bf,group", [(torch.bfloat16, 128, 32, 4), (torch.bfloat16, 64, 10, 4),
                                              (torch.float32, 80, 10, 1), (torch.bfloat16, 128, 32, 8)])
def test_output_in_bf16_is_the_rounded_fp32_output(dtype, d, bf, group, gpu_device):
    from hira_amd.indexer import HIPIndexer
    from hira_amd.searcher import HIPSearcher

    keys, vals = (torch.randn(1, 2, 3000, d, device="cuda").to(dtype) for _ in range(2))
    idx = HIPIndexer(3, 1, bf).build(keys, vals)
    q = torch.randn(2 * group, d, device="cuda").to(dtype)
    tau = torch.full((2 * group,), 2.0, device="cuda") * d ** 0.5
    plan = HIPSearcher().plan_attention(idx, 2 * group, scaling=torch.full((2 * group,), d ** -0.5))
    a = torch.empty(2 * group, d, device="cuda")
    b = torch.empty(2 * group, d, device="cuda", dtype=torch.bfloat16)
    plan.run(q, tau, a)
    plan.run(q, tau, b)
    assert bool((a != 0).any()) and torch.equal(b, a.to(torch.bfloat16))


def _layer(update_every, prompt):
    from hira_amd.cache.hira_cache import HiraCacheLayer
    from hira_amd.cache.hira_config import DeviceMode

    layer = HiraCacheLayer(DeviceMode.CUDA_ONLY, update_every,
                           {"num_levels": 2, "max_iterations": 1, "branching_factor": 32}, {},
                           {"method": "sample_mean_topk", "sample_size": 100, "topk": 4})
    layer.update(prompt, prompt)
    return layer


def _misaligned(x):
    """The same values, contiguous, one element past a 16-byte boundary."""
    y = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:].view(x.shape)
    y.copy_(x)
    assert y.is_contiguous() and y.data_ptr() % 16
    return y


@pytest.mark.parametrize("update_every,m", [(8, 3), (1, 1), (4, 64)])
@pytest.mark.parametrize("form", [_misaligned, lambda x: x.transpose(1, 2).contiguous().transpose(1, 2),
                                  lambda x: x[:, :1].contiguous().expand(x.shape)])
def test_cache_layer_takes_rows_however_they_lie(form, update_every, m, gpu_device):
    """Queue, sample and index are the same from misaligned, strided and expanded (head stride 0)
    tensors as from plain ones."""
    prompt = torch.randn(1, 2, 500, 64, device="cuda").to(torch.bfloat16)
    tokens = torch.randn(6, 1, 2, m, 64, device="cuda").to(torch.bfloat16)
    a = _layer(update_every, prompt.clone())
    b = _layer(update_every, _misaligned(prompt))
    assert torch.equal(a.samples, b.samples)
    for t in tokens:
        x = form(t)
        a.update(x.clone(memory_format=torch.contiguous_format), -x.clone(memory_format=torch.contiguous_format), 0)
        b.update(x, form(-t), 0)
        assert torch.equal(a.queued_keys, b.queued_keys) and torch.equal(a.queued_values, b.queued_values)
        assert torch.equal(a.samples, b.samples)
    a.indexer.sync_sizes(), b.indexer.sync_sizes()
    n = a.indexer.size[0]
    assert torch.equal(a.indexer.perm[:, :n], b.indexer.perm[:, :n])
    assert torch.equal(a.indexer.values_buf[:, :n], b.indexer.values_buf[:, :n])


def test_rows_of_the_wrong_shape_are_refused(gpu_device):
    """Too few heads or columns raise on the host, as a copy of them would; nothing is launched."""
    from hira_amd import _lib
    from hira_amd.indexer import HIPIndexer
    from hira_amd.searcher import HIPSearcher

    prompt = torch.randn(1, 2, 500, 64, device="cuda").to(torch.bfloat16)
    row = prompt[:, :, :1].contiguous()
    for every in (8, 1):
        layer = _layer(every, prompt)
        with pytest.raises((RuntimeError, ValueError)):
            layer.update(row, row[..., :32].contiguous(), 0)
        with pytest.raises((RuntimeError, ValueError)):
            layer.update(row[..., :32].contiguous(), row, 0)
    index = HIPIndexer(2, 1, 32).build(prompt, prompt)
    with pytest.raises((RuntimeError, ValueError)):
        index.update(row, row[..., :32].contiguous())
    q, tau = torch.randn(2, 64, device="cuda").to(torch.bfloat16), torch.zeros(2, device="cuda")
    with pytest.raises((RuntimeError, ValueError)):
        HIPSearcher().search_attention(q, tau, index, queue_keys=prompt[:, :, :8], queue_values=prompt[:, :, :7])
    odd = _misaligned(row)
    with pytest.raises(ValueError):
        _lib.check(_lib.lib().hira_enqueue(prompt.data_ptr(), prompt.data_ptr(), _lib.HIRA_BF16, 2, 500, 0, 1, 64, 64,
                                           odd.data_ptr(), row.data_ptr(), _lib.current_stream(row.device)))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,d", [(1, 1, 64), (3, 3, 72), (4, 1, 128), (40, 32, 128), (40, 33, 64), (600, 50, 64)])
def test_an_append_replaces_members_of_a_sample(dtype, m, n, d, gpu_device):
    """The same index as an append alone, and the sample's rows replaced: key by key, as a window, more rows
    than go with the launch, a window that is grafted."""
    from hira_amd.indexer import HIPIndexer

    k, v = torch.randn(2, 1, 3, 900 + m, d, device="cuda").to(dtype)
    alone, both = (HIPIndexer(3, 1, 16).build(k[:, :, :900], v[:, :, :900]) for _ in range(2))
    sample = torch.randn(3, 70, d, device="cuda").to(dtype)
    slots, which = torch.randperm(70)[:n].tolist(), torch.randint(0, m, (n,)).tolist()
    want = sample.clone()
    want[:, slots] = k[0, :, 900:][:, which]
    alone.update(k[:, :, 900:], v[:, :, 900:])
    both.update(k[:, :, 900:], v[:, :, 900:], sample=(sample, slots, which))
    assert torch.equal(sample, want)
    assert both.size == alone.size
    for a, b in zip([alone.perm, alone.keys_buf, alone.values_buf] + alone.centers[1:] + alone.radii[1:] + alone.counts[1:],
                    [both.perm, both.keys_buf, both.values_buf] + both.centers[1:] + both.radii[1:] + both.counts[1:]):
        assert torch.equal(a, b)
    with pytest.raises(ValueError):
        both.update(k[:, :, 900:], v[:, :, 900:], sample=(sample, [70], [0]))
