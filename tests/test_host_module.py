"""The native host side (csrc/host.cpp) without a GPU: the random numbers it draws, and that what is not the form of a running
program's call is left to the Python body."""
import ctypes as C
import gc
import shutil
import subprocess
import sys
import weakref
from types import SimpleNamespace

import pytest
import torch

from hira_amd import _lib
from hira_amd.attention.hira_attention import hira_attention_forward
from hira_amd.indexer import HIPIndexer
from hira_amd.searcher.hip import DecodePlan


def _draw(gen, m, first, members, seen):
    """Reservoir sampling in torch: the slots of the sample that are replaced, and by which keys."""
    who = [first + i for i, u in enumerate(torch.rand(m, generator=gen).tolist()) if u < members / (seen + i + 1)]
    slots = torch.randint(0, members, (len(who),), generator=gen).tolist() if who else []
    last = dict(zip(slots, who))
    return tuple(last.keys()), tuple(last.values())


@pytest.mark.parametrize("default", [torch.float32, torch.float64, torch.bfloat16, torch.float16])
def test_the_numbers_of_torch(default):
    torch.set_default_dtype(default)
    try:
        a, b = torch.Generator().manual_seed(3), torch.Generator().manual_seed(3)
        for m, first, members, extra in [(1, 0, 1000, 0), (1, 0, 1, 5000), (15, 1, 7, 3), (16, 0, 4096, 10), (700, 2, 33, 100),
                                         (3000, 0, 4096, 1)] * 20:
            assert _lib.host().draw(a, m, first, members, members + extra) == _draw(b, m, first, members, members + extra)
        assert torch.equal(a.get_state(), b.get_state())
    finally:
        torch.set_default_dtype(torch.float32)


@pytest.mark.parametrize("other", ["torch", "commit", "interpreter", "library"])
def test_a_module_built_for_another_is_refused(other, monkeypatch):
    assert _lib.host() is _lib._host_module
    monkeypatch.setattr(_lib, "_host_module", None)
    if other == "torch":
        monkeypatch.setattr(torch, "__version__", "2.10.1")
    elif other == "commit":
        monkeypatch.setattr(torch.version, "git_version", "0" * 40)
    elif other == "interpreter":
        monkeypatch.setattr(_lib, "sys", SimpleNamespace(executable=sys.executable, version_info=(3, 99, 0)))
    else:
        monkeypatch.setattr(_lib, "lib", lambda: SimpleNamespace(hira_abi_version=lambda: _lib.HIRA_ABI_VERSION + 1))
    with pytest.raises(RuntimeError, match="was built for"):
        _lib.host()
    assert _lib._host_module is None


def _tree_with_stand_ins(tmp_path):
    """The Makefile beside empty sources, under an interpreter whose torch is what a file says and a compiler that writes empty files.
    make(*targets) returns how often that has compiled so far."""
    csrc = tmp_path / "hira_amd" / "csrc"
    csrc.mkdir(parents=True)
    shutil.copy(_lib.CSRC / "Makefile", csrc)
    (tmp_path / "include").mkdir()
    for f in (csrc / "host.cpp", tmp_path / "include" / "hira_hip.h", csrc / "libhira_hip.so"):
        f.touch()
    python, cxx = tmp_path / "python", tmp_path / "c++"
    python.write_text(f'#!/bin/sh\ncase "$2" in *EXT_SUFFIX*) echo .tag.so;; *torch*) cat {tmp_path}/torch;; esac\n')
    cxx.write_text(f'#!/bin/sh\necho "$*" >> {tmp_path}/compiled\nwhile [ "$1" != -o ]; do shift; done\ntouch "$2"\n')
    for f in (python, cxx):
        f.chmod(0o755)

    def make(*targets):
        subprocess.run(["make", "-C", str(csrc), f"PYTHON={python}", f"CXX={cxx}", "-o", "libhira_hip.so", *targets], check=True,
                       capture_output=True)
        log = tmp_path / "compiled"
        return len(log.read_text().splitlines()) if log.exists() else 0

    return make


def test_another_torch_is_another_build(tmp_path):
    make = _tree_with_stand_ins(tmp_path)
    (tmp_path / "torch").write_text("2.10.0 abc\n")
    assert make() == 1 and make() == 1 and make("host") == 1
    assert (tmp_path / "hira_amd" / "_host.tag.so").exists()
    (tmp_path / "torch").write_text("2.10.1 abc\n")
    assert make() == 2 and make() == 2
    assert [line.split("HIRA_HOST_TORCH=")[1][:12] for line in (tmp_path / "compiled").read_text().splitlines()] == ['"2.10.0 abc"', '"2.10.1 abc"']


def test_the_library_is_built_without_torch(tmp_path):
    make = _tree_with_stand_ins(tmp_path)
    assert make() == 0
    with pytest.raises(subprocess.CalledProcessError):
        make("host")
    (tmp_path / "torch").write_text("2.10.0 abc\n")
    assert make() == 1


def test_what_is_not_the_form_is_left_alone():
    host = _lib.host()
    q, k, v = torch.zeros(1, 2, 4, 16), torch.zeros(1, 2, 1, 16), torch.zeros(1, 2, 1, 16)
    assert host.enqueue(q, q.clone(), k, v, 0, 0, 0) is None  # (host memory)
    assert host.enqueue(None, q, k, [1], 0, 0, 0) is None
    tree, query, out, launch = _lib.HiraTree(num_trees=2, dim=16, vdim=16), _lib.HiraQuery(4), _lib.HiraSearchOut(), _lib.HiraLaunch()
    sample, queue, ws, tau = _lib.HiraSample(), _lib.HiraQueue(), torch.zeros(64, dtype=torch.uint8), torch.zeros(4)
    at = *(C.addressof(x) for x in (tree, query, sample, queue, out, launch)), 0, ws, 64, 1
    assert host.attend(at, tau, torch.zeros(1, 4, 1, 16), torch.zeros(2, 8, 16), q, q, 1, 0, 1, 0) is None
    at = C.addressof(tree), C.addressof(query), C.addressof(out), 4, 0, 1
    assert host.search(at, C.addressof(launch), torch.zeros(4, 16), tau, None, torch.zeros(4, 8), 0.0, 0) is None
    assert host.append(C.addressof(tree), k, v, 1, 0, None, (), (), 0, 0, None, 0) is None
    assert query.q is None and out.attn_out is None and out.dense is None
    for name in ("enqueue", "attend", "search", "append", "draw"):
        with pytest.raises(TypeError):
            getattr(host, name)(1)
    with pytest.raises(TypeError):
        host.draw(3, 1, 0, 1, 1)
    with pytest.raises(ValueError):
        host.draw(torch.Generator(), 1, 0, 0, 1)


class _Structs:
    """An index as far as a plan looks at it when its level sizes may have moved."""

    device = torch.device("cpu")

    def __init__(self):
        self._tree_struct = _lib.HiraTree()

    def tree_struct(self):
        return self._tree_struct


def _plan(monkeypatch, attend, kind=DecodePlan):
    """A plan whose native call is `attend`."""
    monkeypatch.setattr(_lib, "host", lambda: SimpleNamespace(attend=attend))
    monkeypatch.setattr(_lib, "stream_of", lambda dev: 0)
    plan = kind.__new__(kind)
    plan.indexer = _Structs()
    plan.tree, plan.query, plan.sample, plan.queue = plan.indexer._tree_struct, _lib.HiraQuery(4), _lib.HiraSample(), _lib.HiraQueue()
    plan.out, plan.launch, plan._at, plan._dev = _lib.HiraSearchOut(), _lib.HiraLaunch(), None, 0
    plan.tau_buf, plan.ws, plan.ws_bytes, plan._ws_rows = torch.zeros(4), torch.zeros(64, dtype=torch.uint8), 64, 1
    plan._workspace_need = lambda: 64
    return plan


def test_a_plan_holds_its_structs_while_the_call_reads_them(monkeypatch):
    """The call lets other threads run: one of them may be the first to see that the index moved."""
    trees = []

    def attend(at, *rest):
        trees.append(weakref.ref(plan.tree))
        assert at[0] == C.addressof(plan.tree) and at[1] == C.addressof(plan.query)
        plan.indexer._tree_struct = _lib.HiraTree()
        plan._follow_index()
        gc.collect()
        assert trees[-1]() is not None and C.addressof(trees[-1]()) == at[0]
        return rest[1]

    plan = _plan(monkeypatch, attend)
    for _ in range(3):
        assert plan.attend("query", None, "sample_mean_topk", 3, None, None, 0) == "query"
        plan._at = None
        gc.collect()
        assert trees[-1]() is None


def test_a_plan_whose_tree_is_replaced_while_it_looks_up_the_addresses(monkeypatch):
    plan = _plan(monkeypatch, lambda at, *rest: at)
    plan.attend(None, None, "sample_mean_topk", 3, None, None, 0)
    stale = plan._at
    plan.indexer._tree_struct = _lib.HiraTree()
    plan._follow_index()
    plan._at = stale  # (what a thread that had looked before leaves behind)
    assert plan.attend(None, None, "sample_mean_topk", 3, None, None, 0)[0] == C.addressof(plan.tree)


def _ones(self, query, samples, method, k, out, *rest):
    out.fill_(1.0)


class _OwnStep(DecodePlan):
    run_sampled = _ones


@pytest.mark.parametrize("how", ["a subclass's", "the plan's", "the class's", "no attend"])
def test_a_plan_that_takes_its_step_another_way(how, monkeypatch):
    """The attention function calls run_sampled where it is not the one that the native call stands for."""
    plan = _plan(monkeypatch, lambda *a: torch.zeros(1, 1, 4, 16), _OwnStep if how == "a subclass's" else DecodePlan)
    ix = plan.indexer
    ix.keys_buf, ix.dtype, ix.vdim, ix.num_trees = torch.zeros(2, 32, 16), torch.float32, 16, 2
    q = torch.zeros(1, 4, 1, 16)
    rows = torch.zeros(1, 2, 8, 16)
    cache = SimpleNamespace(prefill_keys=None, indexer=ix, searcher=SimpleNamespace(decode_plan=lambda *a: plan), samples=torch.zeros(2, 8, 16),
                            threshold_method="sample_mean_topk", threshold_topk=3, queue_rows=2, queue_store=(rows, rows))
    if how != "a subclass's":
        assert torch.equal(hira_attention_forward(None, q, cache, None, scaling=1.0)[0], torch.zeros(1, 1, 4, 16))
    if how == "the plan's":
        plan.run_sampled = _ones.__get__(plan)
    elif how == "the class's":
        monkeypatch.setattr(DecodePlan, "run_sampled", _ones)
    elif how == "no attend":
        plan = SimpleNamespace(run_sampled=lambda *a: _ones(None, *a))
    assert torch.equal(hira_attention_forward(None, q, cache, None, scaling=1.0)[0], torch.ones(1, 1, 4, 16))


@pytest.mark.parametrize("code,late,added", [(-2, False, 0), (-1, False, 0), (-2, True, 3), (-1, True, 3)])
def test_an_append_whose_sizes_could_not_be_read_back(code, late, added, monkeypatch):
    """The keys count as soon as their rows are in, and the error is the read-back's; rows that something may yet write into are
    not used again."""
    behind = _lib.host().APPENDED
    monkeypatch.setattr(_lib, "host", lambda: SimpleNamespace(append=lambda *a: code - late * behind, APPENDED=behind))
    monkeypatch.setattr(_lib, "stream_of", lambda dev: 0)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    ix = HIPIndexer(2, 0, 16, device="cpu")
    ix.batch, ix.num_heads, ix.num_trees, ix.dim, ix.vdim, ix.num_keys, ix.tiled = 1, 2, 2, 16, 16, 40, False
    ix.keys_buf = ix.values_buf = SimpleNamespace(get_device=lambda: 0)
    ix._state = torch.zeros(2, 10, dtype=torch.int32)
    ix._needed_caps, ix._grow, ix.tree_struct = lambda m: None, lambda need: None, _lib.HiraTree
    ix._rows_to_read_into = lambda n: torch.zeros(n, dtype=torch.int64)
    ix._host_rows = kept = torch.zeros(20, dtype=torch.int64)
    rows = torch.zeros(1, 2, 3, 16)
    with pytest.raises(ValueError if code == -1 else RuntimeError):
        ix.update(rows, rows)
    assert ix.num_keys == 40 + added and ix._host_rows is kept
