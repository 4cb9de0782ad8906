"""Calls in the form that the native host side takes against the same calls in other forms (strides, types, storage that is not
aligned), which go through the Python bodies: same results."""
import ctypes as C

import pytest
import torch

from hira_amd import _lib
from hira_amd.attention.hira_attention import hira_attention_forward
from hira_amd.cache.hira_cache import HiraCacheLayer
from hira_amd.indexer import HIPIndexer
from hira_amd.searcher import HIPSearcher

pytestmark = pytest.mark.gpu


def _gen(seed):
    g = torch.Generator().manual_seed(seed)
    return lambda *shape, dtype=torch.bfloat16: torch.randn(shape, generator=g).to(dtype).cuda()


def _strided(x):
    """The same numbers a column of gaps apart."""
    wide = torch.zeros(x.shape[:-1] + (2 * x.shape[-1],), dtype=x.dtype, device=x.device)
    wide[..., ::2] = x
    return wide[..., ::2]


def _misaligned(x):
    flat = torch.zeros(x.numel() + 1, dtype=x.dtype, device=x.device)
    flat[1:] = x.reshape(-1)
    return flat[1:].view(x.shape)


FORMS = {"ready": lambda x: x, "strided": _strided, "misaligned": _misaligned, "fp32": lambda x: x.float(),
         "parameter": lambda x: torch.nn.Parameter(x, requires_grad=False)}


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("every,n", [(4, 300), (1, 300), (3, 900)])
def test_a_decode_through_the_cache_layer(form, every, n, gpu_device):
    as_query = FORMS[form] if form in ("strided", "misaligned", "parameter") else FORMS["ready"]

    def run(form):
        print(f"case form={form} every={every} n={n}", flush=True)
        x = _gen(n + every)
        layer = HiraCacheLayer("cuda_only", every, dict(num_levels=3, max_iterations=1, branching_factor=16), {},
                               dict(method="sample_mean_topk", sample_size=500, topk=7))
        layer.update(x(1, 2, n, 64), x(1, 2, n, 64))
        outs, module = [], type("M", (), {"scaling": 0.125})()
        for _ in range(9):
            k, v, q = FORMS[form](x(1, 2, 1, 64)), FORMS[form](x(1, 2, 1, 64)), x(1, 8, 1, 64)
            held, _ = layer.update(k, v)
            outs.append(hira_attention_forward(module, as_query(q), held, None)[0].clone())
        return torch.cat(outs), layer

    want, a = run("ready")
    got, b = run(form)
    assert torch.equal(want, got) and torch.equal(a.samples, b.samples)
    assert torch.equal(a.queued_keys, b.queued_keys) and torch.equal(a.queued_values, b.queued_values)
    assert torch.equal(a.indexer.keys_buf, b.indexer.keys_buf) and torch.equal(a.indexer.perm, b.indexer.perm)
    assert a.queued_len == b.queued_len and a.indexer.num_keys == b.indexer.num_keys


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_search_like_one_before_it(dtype, gpu_device):
    x = _gen(5)
    index = HIPIndexer(3, 1, 16).build(x(1, 2, 900, 64, dtype=dtype))
    tau, sc = torch.tensor([3.0, 5.0, 8.0, 2.0]).cuda(), torch.tensor([1.0, 0.5, 2.0, 4.0]).cuda()
    kept = HIPSearcher(output_fill_value=-7.0)

    def fresh():
        return HIPSearcher(output_fill_value=kept.output_fill_value, kernel=kept.launch.kernel)

    for step in range(3):
        q = x(4, 64, dtype=dtype)
        for query in (q, q[None, :, None], _strided(q), _misaligned(q), q.double()):
            for t, s in ((tau, None), (tau, sc), (4.0, None), (tau.double(), _strided(sc)), (_strided(tau), sc)):
                assert torch.equal(kept.search(query, t, index, scaling=s), fresh().search(query, t, index, scaling=s))
        assert torch.equal(kept.search(q[:2], tau[:2], index), fresh().search(q[:2], tau[:2], index))  # (other heads)
        kept.output_fill_value += 1.5
        if step == 0:
            index.update(x(1, 2, 40, 64, dtype=dtype))  # (level sizes that moved)
        else:
            kept.launch = HIPSearcher(kernel=1).launch


@pytest.mark.parametrize("form", ["strided", "misaligned", "fp32", "parameter"])
@pytest.mark.parametrize("m", [1, 40])
def test_an_append_and_its_read_back(form, m, gpu_device):
    def run(form):
        x = _gen(m)
        index = HIPIndexer(3, 1, 16).build(x(1, 2, 700, 64), x(1, 2, 700, 64))
        sizes = []
        for _ in range(4):
            index.update(FORMS[form](x(1, 2, m, 64)), FORMS[form](x(1, 2, m, 64)))
            sizes.append(list(index.size))
        index.update(FORMS[form](x(1, 2, 3, 64)), FORMS[form](x(1, 2, 3, 64)))
        return index, sizes

    (a, want), (b, got) = run("ready"), run(form)
    assert want == got and a.size == b.size and a.num_keys == b.num_keys == 700 + 4 * m + 3
    for l in range(1, 3):
        assert torch.equal(a.radii[l], b.radii[l]) and torch.equal(a.counts[l], b.counts[l])
    assert torch.equal(a.perm[:, :a.size[0]], b.perm[:, :b.size[0]]) and torch.equal(a.values_buf[:, :700], b.values_buf[:, :700])
    assert a._host_rows is not None and b._host_rows is not None


class _Calls:
    """The native functions' calls with every argument in the form that they take, over stand-ins for the library's functions:
    what they would launch is noted and not done.  `args[name]` may be changed before `call(name)`."""

    def __init__(self):
        self.host, self.launched, self.codes = _lib.host(), [], {}
        x, t, dev = _gen(1), 2, torch.cuda.current_device()
        self.tree = _lib.HiraTree(num_trees=t, num_levels=2, bf=16, dim=64, vdim=32, dtype=_lib.HIRA_BF16)
        self.tree.size[0] = 96
        self.query, self.out, self.queue = _lib.HiraQuery(4), _lib.HiraSearchOut(), _lib.HiraQueue()
        self.sample, self.launch = _lib.HiraSample(), _lib.HiraLaunch()
        at = {n: C.addressof(getattr(self, n)) for n in ("tree", "query", "sample", "queue", "out", "launch")}
        self.state, one = torch.zeros(t, 10, dtype=torch.int32, device="cuda"), torch.ones(4, device="cuda")
        self.keep = one
        k, v, samples = x(1, t, 1, 64), x(1, t, 1, 32), x(t, 40, 64)
        qk, qv = x(1, t, 8, 64), x(1, t, 8, 32)
        back = torch.zeros(t * (_lib.HIRA_MAX_LEVELS + 2), dtype=torch.int64, pin_memory=True)
        self.args = {
            "enqueue": [qk, qv, k, v, 3, dev, 0],
            "attend": [(*at.values(), dev, torch.zeros(512, dtype=torch.uint8, device="cuda"), 512, 8), one.clone(), x(1, 4, 1, 64), samples,
                       qk, qv, 5, 1, 3, 0],
            "search": [(at["tree"], at["query"], at["out"], 4, dev, one.data_ptr()), at["launch"], x(4, 64), one.clone(), one.clone(),
                       torch.zeros(4, 96, device="cuda"), -7.0, 0],
            "append": [at["tree"], x(1, t, 3, 64), x(1, t, 3, 32), 3, self.state.data_ptr(), samples, (4, 0), (1, 2), dev, 0, back, 1],
        }

    def __enter__(self):
        def stand_in(name):
            res, args = _lib.SYMBOLS[name]
            return C.CFUNCTYPE(res, *args)(lambda *a: self.launched.append(name) or self.codes.get(name, 0))

        self.functions = {name: stand_in(name) for name in ("hira_enqueue", "hira_search", "hira_search_sampled", "hira_update_sample",
                                                            "hira_read_state")}
        self.host.bind({name: C.cast(f, C.c_void_p).value for name, f in self.functions.items()})
        return self

    def __exit__(self, *exc):
        lib = _lib.lib()
        self.host.bind({name: C.cast(getattr(lib, name), C.c_void_p).value for name in _lib.SYMBOLS})

    def call(self, name):
        """(what came back, what was launched, were the structs changed)"""
        structs = self.query, self.out, self.queue, self.sample
        before, n = [bytes(s) for s in structs], len(self.launched)
        result = getattr(self.host, name)(*self.args[name])
        return result, self.launched[n:], [bytes(s) for s in structs] != before

    def refused(self, name):
        result, launched, changed = self.call(name)
        return result is None and not launched and not changed


CHUNKS = [("enqueue", 0), ("enqueue", 1), ("enqueue", 2), ("enqueue", 3), ("attend", 2), ("attend", 3), ("attend", 4), ("attend", 5),
          ("search", 2), ("append", 1), ("append", 2), ("append", 5)]


@pytest.mark.parametrize("name,i", CHUNKS)
def test_rows_that_start_between_two_chunks_are_left_alone(name, i, gpu_device):
    with _Calls() as calls:
        assert calls.call(name)[1]
        calls.args[name][i] = _misaligned(calls.args[name][i])
        assert calls.refused(name)
        if name == "append" and i < 3:  # (without a sample too)
            calls.args[name][5:8] = None, (), ()
            assert calls.refused(name)


def _to(i, value):
    return lambda args: args.__setitem__(i, value(args[i]) if callable(value) else value)


def _part(i, value):
    """A part of the first argument."""
    return _to(0, lambda at: (*at[:i], value(at[i]) if callable(value) else value, *at[i + 1:]))


def _rows(*shape, dtype=torch.bfloat16):
    return lambda old: torch.zeros(shape, dtype=dtype, device="cuda")


BIG = 2 ** 31
WRONG = {
    "enqueue": {
        "a full queue": _to(4, 8), "before the queue": _to(4, -1), "two rows": _to(2, _rows(1, 2, 2, 64)), "more heads": _to(2, _rows(1, 3, 1, 64)),
        "more sequences": _to(3, _rows(2, 2, 1, 32)), "narrow keys": _to(2, _rows(1, 2, 1, 32)), "wide values": _to(3, _rows(1, 2, 1, 64)),
        "another type": _to(3, _rows(1, 2, 1, 32, dtype=torch.float32)), "a shorter queue of values": _to(1, _rows(1, 2, 7, 32)),
        "a queue of fewer heads": _to(1, _rows(1, 1, 8, 32)), "three dimensions": _to(2, _rows(2, 1, 64)), "half precision": _to(0, _rows(1, 2, 8, 64, dtype=torch.float16)),
        "strided": _to(2, _strided), "host memory": _to(2, lambda x: x.cpu()), "another device": _to(5, lambda d: d + 1), "no tensor": _to(3, None)},
    "attend": {
        "more rows than the queue holds": _to(6, 9), "more rows than the workspace is for": _part(9, 4), "rows below none": _to(6, -1),
        "rows that are no number": _to(6, 5.0), "a workspace that is too small": _part(8, 513), "a workspace of numbers": _part(7, _rows(512, dtype=torch.float32)),
        "few thresholds": _to(1, _rows(3, dtype=torch.float32)), "thresholds in 16 bits": _to(1, _rows(4)), "more heads": _to(2, _rows(1, 5, 1, 64)),
        "two positions": _to(2, _rows(1, 2, 2, 64)), "a wide query": _to(2, _rows(1, 4, 1, 128)), "a query in fp32": _to(2, lambda x: x.float()),
        "samples of three trees": _to(3, _rows(3, 40, 64)), "narrow samples": _to(3, _rows(2, 40, 32)), "samples in fp32": _to(3, lambda x: x.float()),
        "a queue of three trees": _to(4, _rows(1, 3, 8, 64)), "a queue of wide keys": _to(4, _rows(1, 2, 8, 128)), "a longer queue of values": _to(5, _rows(1, 2, 9, 32)),
        "a queue of wide values": _to(5, _rows(1, 2, 8, 64)), "values of one tree": _to(5, _rows(1, 1, 8, 32)), "no queue": _to(4, None),
        "a large k": _to(8, BIG), "a k that is no number": _to(8, 3.0), "five structs": _to(0, lambda at: at[1:]), "strided": _to(2, _strided)},
    "search": {
        "more heads": _to(2, _rows(5, 64)), "a wide query": _to(2, _rows(4, 128)), "as many numbers in wider rows": _to(2, _rows(2, 128)),
        "a query in fp32": _to(2, lambda x: x.float()), "two positions": _to(2, _rows(1, 2, 2, 64)), "few thresholds": _to(3, _rows(3, dtype=torch.float32)),
        "thresholds in 16 bits": _to(3, _rows(4)), "a number": _to(3, 4.0), "few scales": _to(4, _rows(2, dtype=torch.float32)), "scales in 64 bits": _to(4, lambda x: x.double()),
        "fewer slots": _to(5, _rows(4, 95, dtype=torch.float32)), "more slots": _to(5, _rows(4, 97, dtype=torch.float32)), "fewer rows": _to(5, _rows(3, 96, dtype=torch.float32)),
        "an output in 16 bits": _to(5, _rows(4, 96)), "five structs": _to(0, lambda at: at[:5]), "strided": _to(2, _strided)},
    "append": {
        "fewer rows": _to(3, 2), "more rows": _to(3, 4), "rows below none": _to(3, -3), "values of more rows": _to(2, _rows(1, 2, 4, 32)), "wide values": _to(2, _rows(1, 2, 3, 64)),
        "keys in fp32": _to(1, lambda x: x.float()), "values in fp32": _to(2, lambda x: x.float()), "a sample of three trees": _to(5, _rows(3, 40, 64)),
        "a narrow sample": _to(5, _rows(2, 40, 32)), "a sample in fp32": _to(5, lambda x: x.float()), "a flat sample": _to(5, _rows(80, 64)),
        "more slots than keys": _to(6, (1, 2, 3)), "slots in a list": _to(6, [4, 0]), "a large slot": _to(6, (BIG, 0)), "a slot that is no number": _to(6, (4.0, 0)),
        "a very large key": _to(7, (1, 2 ** 70)), "few rows to read into": _to(10, lambda r: r[:-1]), "rows of half the size": _to(10, lambda r: r.int()),
        "rows on the device": _to(10, lambda r: r.cuda()), "strided": _to(1, _strided), "another device": _to(8, lambda d: d + 1)},
}


@pytest.mark.parametrize("name,wrong", [(name, wrong) for name in WRONG for wrong in WRONG[name]])
def test_what_is_not_the_form_is_left_alone(name, wrong, gpu_device):
    """One property off: None, nothing launched, nothing changed."""
    with _Calls() as calls:
        result, launched, changed = calls.call(name)
        assert launched and result is not None
        WRONG[name][wrong](calls.args[name])
        assert calls.refused(name)


def test_what_the_library_answers_comes_back(gpu_device):
    with _Calls() as calls:
        assert calls.call("enqueue")[:2] == (0, ["hira_enqueue"]) and calls.call("search")[:2] == (0, ["hira_search"])
        out, launched, changed = calls.call("attend")
        assert launched == ["hira_search_sampled"] and changed and out.shape == (1, 1, 4, 32) and calls.out.attn_out == out.data_ptr()
        assert (calls.queue.len, calls.queue.cap, calls.sample.num_rows, calls.sample.k) == (5, 8, 40, 3)
        back, launched, _ = calls.call("append")
        assert launched == ["hira_update_sample", "hira_read_state"] and len(back) == _lib.HIRA_MAX_LEVELS + 2
        for function in ("hira_enqueue", "hira_search", "hira_search_sampled", "hira_read_state"):
            calls.codes[function] = -2
        assert calls.call("enqueue")[0] == calls.call("search")[0] == calls.call("attend")[0] == -2
        assert calls.call("append")[0] == -2 - calls.host.APPENDED
        calls.codes["hira_update_sample"] = -1
        assert calls.call("append")[:2] == (-1, ["hira_update_sample"])
