"""An index in host memory: restored, adopted, grown and saved without a GPU; what would launch a kernel
on it is refused."""
import copy
import pickle

import numpy as np
import pytest
import torch

from hira_amd import _lib
from hira_amd.indexer.hip import HIPIndexer
from oracle import hira_oracle as ho


def _parts(dtype, bf=16, n=300, d=64, trees=2, seed=0):
    rng = np.random.default_rng(seed)
    keys = torch.from_numpy(rng.normal(size=(trees, n, d)).astype(np.float32)).to(dtype).float().numpy()
    size = ho.fixed_fanout_sizes(n, bf, 3)
    pad, perm = np.zeros((trees, size[0], d), np.float32), np.full((trees, size[0]), -1, np.int32)
    pad[:, :n], perm[:, :n] = keys, np.arange(n)
    k1, k2 = size[1], size[2]
    counts1 = np.clip(n - np.arange(k1) * bf, 0, bf).astype(np.int32)
    c1, c2 = (rng.normal(size=(trees, k, d)).astype(np.float32) for k in (k1, k2))
    return dict(bf=bf, keys=pad, perm=perm, values=pad.copy(), dtype=dtype, centers=[None, c1, c2],
                radii=[None, np.full((trees, k1), 20.0, np.float32), np.full((trees, k2), 40.0, np.float32)],
                counts=[None, np.tile(counts1, (trees, 1)), np.full((trees, k2), bf, np.int32)])


@pytest.mark.parametrize("dtype,layout", [(torch.float32, "row_major"), (torch.bfloat16, "row_major"),
                                          (torch.bfloat16, "tiled")])
@pytest.mark.parametrize("capacity", [None, 2000])
def test_adopted_saved_loaded_and_grown(dtype, layout, capacity, tmp_path):
    p = _parts(dtype)
    a = HIPIndexer.from_layout(device="cpu", layout=layout, capacity=capacity, **p)
    n = a.size[0]
    keys = torch.from_numpy(p["keys"]).to(dtype)

    def whole(x):
        assert x.size == a.size and x.num_keys == 300 and all(c >= s for c, s in zip(x.cap, x.size))
        assert torch.equal(x.keys_rowmajor(), keys) and torch.equal(x.values_buf[:, :n], keys)
        assert torch.equal(x.perm[:, :n], torch.from_numpy(p["perm"]))
        for l in (1, 2):
            k = x.size[l]
            assert torch.equal(x.centers_rowmajor(l), torch.from_numpy(p["centers"][l]).to(dtype))
            assert torch.equal(x.radii[l][:, :k], torch.from_numpy(p["radii"][l]))
            assert torch.equal(x.counts[l][:, :k], torch.from_numpy(p["counts"][l]))
            # what lies behind the slots in use is empty
            assert bool((x.radii[l][:, k:] == float("-inf")).all()) and not x.counts[l][:, k:].any()
        assert bool((x.perm[:, n:] == -1).all()) and not x.values_buf[:, n:].any()

    whole(a)
    path = str(tmp_path / "index.safetensors")
    a.save(path)
    b = HIPIndexer.load(path, device="cpu", capacity=capacity)
    whole(b)
    b.reserve(5000)
    assert b.cap[0] > n + 5000 - 300
    whole(b)
    b.begin_unsynced(10)
    assert b._state.shape == (2, _lib.HIRA_MAX_LEVELS + 2)
    assert b._state[0].tolist()[:3] == [0, a.size[1], a.size[2]] and int(b._state[1, _lib.HIRA_MAX_LEVELS]) == 300


def test_no_kernel_is_launched_over_host_memory():
    p = _parts(torch.float32)
    a = HIPIndexer.from_layout(device="cpu", layout="row_major", **p)
    new = torch.zeros((1, 2, 1, 64))
    for call in (lambda: a.update(new, new), lambda: HIPIndexer(2, device="cpu").build(new, new),
                 lambda: HIPIndexer.from_layout(device="cpu", layout="q8", **_parts(torch.bfloat16))):
        with pytest.raises(ValueError, match="GPU"):
            call()
    with pytest.raises(ValueError, match="GPU"):
        _lib.stream_of(-1)
    with pytest.raises(ValueError, match="GPU"):
        _lib.current_stream(torch.device("cpu"))


def test_no_search_is_launched_over_host_memory():
    from hira_amd.searcher.hip import HIPSearcher

    a = HIPIndexer.from_layout(device="cpu", layout="row_major", **_parts(torch.float32))
    q, tau = torch.zeros((4, 64)), torch.zeros((4,))
    for call in (HIPSearcher().search, HIPSearcher().search_attention, HIPSearcher().search_compact):
        for scaling in (None, torch.ones(4)):
            with pytest.raises(ValueError, match="GPU"):
                call(q, tau, a, scaling=scaling)


def test_a_plans_workspace_goes_by_the_queued_rows_in_use():
    """Few rows in a large buffer take no workspace for all of it; a queue that fills up has a new one made
    a few times only."""
    from hira_amd.searcher.hip import HIPSearcher

    a = HIPIndexer.from_layout(device="cpu", layout="row_major", **_parts(torch.float32))

    def plan():
        return HIPSearcher().plan_attention(a, 8, scaling=torch.ones(8))

    q, out = torch.zeros((8, 64)), torch.zeros((8, 64))
    large, small = (torch.empty((2, 1, 64)).expand(2, cap, 64) for cap in (1 << 20, 1024))
    few, whole, filled = plan(), plan(), plan()
    few._step(q, out, large, large, 3)
    whole._step(q, out, small, small, 1024)
    assert few.ws_bytes <= whole.ws_bytes
    made = 0
    for m in range(1, 1025):
        before = filled.ws_bytes
        filled._step(q, out, small, small, m)
        made += filled.ws_bytes != before
        assert filled._ws_rows >= m
    assert made <= 4 and filled.ws_bytes == whole.ws_bytes


def test_sizes_are_read_back_with_the_indexs_device_current(monkeypatch):
    """sync_sizes() and save() take an index on any device, whichever is current."""
    import contextlib
    from types import SimpleNamespace

    a = HIPIndexer.from_layout(device="cpu", layout="row_major", **_parts(torch.float32))
    n = 2 * (_lib.HIRA_MAX_LEVELS + 2)
    a._state = SimpleNamespace(is_cuda=True, get_device=lambda: 1, data_ptr=lambda: 0, numel=lambda: n)
    a._host_rows, a._pending = torch.zeros(n, dtype=torch.int64), 1
    current = [0]

    @contextlib.contextmanager
    def device(index):
        current.append(index)
        yield
        current.pop()

    def read(tree, state, rows, ticket, most, stream):
        assert current[-1] == 1 and stream == 7
        most[1], most[2] = a.size[1], a.size[2]
        return 0

    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: current[-1])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(_lib, "stream_of", lambda index: 7)
    monkeypatch.setattr(_lib, "lib", lambda: SimpleNamespace(hira_read_state=read))
    a.sync_sizes()
    assert a._pending == 0 and current == [0]


def test_a_copied_index_has_pointers_and_pinned_rows_of_its_own():
    a = HIPIndexer.from_layout(device="cpu", layout="row_major", **_parts(torch.float32))
    a._host_rows, at = torch.zeros(20, dtype=torch.int64), a.tree_struct().keys
    for b in (copy.deepcopy(a), pickle.loads(pickle.dumps(a))):
        assert b._host_rows is None and b._append is None
        assert b.tree_struct().keys == b.keys_buf.data_ptr() != at
        assert torch.equal(b.keys_rowmajor(), a.keys_rowmajor()) and b.size == a.size
    assert a.tree_struct().keys == at and a._host_rows is not None


def test_a_read_back_has_rows_of_its_own_while_it_lasts(monkeypatch):
    """Two threads may ask for an index's sizes at once: neither call's rows or ticket are the other's, and one set of
    rows is kept."""
    from types import SimpleNamespace

    a = HIPIndexer.from_layout(device="cpu", layout="row_major", **_parts(torch.float32))
    n = 2 * (_lib.HIRA_MAX_LEVELS + 2)
    a._state = SimpleNamespace(is_cuda=True, get_device=lambda: 0, data_ptr=lambda: 0, numel=lambda: n)
    a._host_rows, zeros, seen = torch.zeros(n, dtype=torch.int64), torch.zeros, []

    def read(tree, state, rows, ticket, most, stream):
        seen.append((rows, ticket))
        if len(seen) == 1:  # (while the first call waits)
            a._largest_state()
        most[:] = range(len(most))
        return 0

    monkeypatch.setattr(torch, "zeros", lambda *args, pin_memory=False, **kw: zeros(*args, **kw))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(_lib, "stream_of", lambda index: 0)
    monkeypatch.setattr(_lib, "lib", lambda: SimpleNamespace(hira_read_state=read))
    assert a._largest_state() == list(range(n // 2))
    a._largest_state()
    assert len(seen) == 3 and len({t for _, t in seen}) == 3 and seen[0][0] != seen[1][0]
    assert seen[2][0] == seen[0][0] == a._host_rows.data_ptr()
