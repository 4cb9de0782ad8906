"""HIPSearcher: halfspace range search (and fused sparse attention) on one MI355X.

Replaces the reference's GPU searcher (searcher/cuda.py:15-143) and, through
``index_space="position"``, the CPU searcher's contract (searcher/cpu.py:44-101):
``search(query (1,H_q,1,D), threshold (H_q,), indexer, q_head_to_kv=None, scaling=None)``
returns an ``(H_q, N)`` fp32 tensor holding ``score * scaling`` for every key with
``q.k >= threshold`` and ``output_fill_value`` elsewhere.

Semantics follow the CPU kernels (keep a node when ``q.c + ||q|| r >= t``, a key when
``q.k >= t``: kernels/cpp/torch_ext_v3.cpp:182, 212, 238), not the Triton kernels, which
gate with a strict ``>`` and never filter the leaves (kernels/triton_search_kernels.py:
49-63).  Like the reference's GPU searcher the dense result lives in a buffer this object
keeps and reuses: clone it to hold on to a result across calls (searcher/cuda.py:35-54).
"""
from __future__ import annotations

import ctypes as C
from threading import get_ident
from typing import Optional, Tuple

import torch

from .. import _lib
from .base import BaseSearcher

DEFAULT_OUTPUT_FILL_VALUE = 0.0

# The workspace's first bytes hold nothing but arrival counters, zero between calls, whatever index a
# call is on: its counters end where this part ends (16384 trees x passes of heads).
_COUNTERS = 64 * 1024


def _on(t: torch.Tensor, device) -> bool:
    """Is tensor `t` on `device`?  ("cuda" without an index means the current device, which a
    tensor's own device always spells out.)"""
    device = torch.device(device)
    if t.device.type != device.type:
        return False
    if device.index is None:
        return device.type != "cuda" or t.device.index == torch.cuda.current_device()
    return t.device.index == device.index


_OUT_TYPES = {torch.float32: _lib.HIRA_F32, torch.bfloat16: _lib.HIRA_BF16}


def _refuse_out(out: torch.Tensor):
    raise ValueError(f"out is {out.dtype}: attention is written as float32, or rounded once to bfloat16")


def _out_type(out: torch.Tensor, numel: int, dev: int) -> int:
    """The type that attention is written to `out` in; ValueError where it cannot be written there."""
    if out.dtype not in _OUT_TYPES:
        _refuse_out(out)
    if out.numel() < numel or out.get_device() != dev or not out.is_contiguous():
        raise ValueError(f"out {tuple(out.shape)} on {out.device}: expected {numel} numbers or more, contiguous, "
                         "on the index's device")
    return _OUT_TYPES[out.dtype]


class _Call:
    """What a call on one tree with one number of heads needs and does not change from call to
    call: the C structs (only this thread fills them in), the head map, the address of a scale of one
    per head (the library's own; None: not asked for yet), the workspace's size.  Made on first use and
    kept by the searcher: a call that comes with ready tensors (the storage type, on the index's device,
    contiguous) then allocates and copies nothing and its host side is a handful of attribute reads
    around one library call (25 -> 11 us for ``search_attention``, which the kernels of small indexes are shorter
    than), and for ``search`` one call of the native host side (21 -> 8 -> 4.6 us, the launch's own time).  That holds from the second call on a tree whose level
    sizes stay: the first on an index, and the first after an append that moved them, makes it anew."""

    __slots__ = ("tree", "query", "out", "queue", "dev", "keep", "ones", "ws_bytes", "ws_at", "ws_for",
                 "launch", "tree_ref", "query_ref", "out_ref", "queue_ref", "launch_ref", "launch_at", "at")

    def __init__(self, tree, query, dev, keep):
        self.tree, self.query, self.dev, self.keep, self.ones = tree, query, dev, keep, None
        self.out = _lib.HiraSearchOut()
        self.queue = _lib.HiraQueue()
        # the workspace and the place in it; the queue rows and launch options it is for
        self.ws_bytes, self.ws_at, self.ws_for = 0, 0, (-1, b"")
        self.tree_ref, self.query_ref = C.byref(tree), C.byref(query)
        self.out_ref, self.queue_ref = C.byref(self.out), C.byref(self.queue)
        self.launch = self.launch_ref = self.launch_at = None
        self.at: Optional[tuple] = None  # what the native search takes of it

    def follow_launch(self, launch) -> None:
        """The searcher's launch options as they are now (callers may replace them, or change their fields)."""
        self.launch, self.launch_ref, self.launch_at = launch, C.byref(launch), C.addressof(launch)

    def addresses(self) -> tuple:
        """(not kept before the scale of ones is known: it is asked for once)"""
        at = (C.addressof(self.tree), C.addressof(self.query), C.addressof(self.out), self.query.num_q_heads, self.dev, self.ones)
        if self.ones:
            self.at = at
        return at


class HIPSearcher(BaseSearcher):
    _MAX_CALLS = 256  # kept call descriptions: a model's layers, several threads, a few growths

    def __init__(self, block_c=None, output_fill_value: float = DEFAULT_OUTPUT_FILL_VALUE,
                 *, index_space: str = "slot", block_threads: int = 0, nodes_per_wave: int = 0,
                 kernel: int = 0, separate_merge: bool = False):
        super().__init__()
        if index_space not in ("slot", "position"):
            raise ValueError("index_space must be 'slot' or 'position'")
        self.block_c = block_c  # accepted for HiraConfig.get_searcher_kwargs(); unused
        self.output_fill_value = float(output_fill_value)
        self.index_space = index_space
        self.launch = _lib.HiraLaunch(int(block_threads), int(nodes_per_wave), int(kernel),
                                      int(bool(separate_merge)))
        self._tmp_out: Optional[torch.Tensor] = None
        self._map_cache = {}
        self._workspace: Optional[torch.Tensor] = None
        self._decode_plans: dict = {}
        self._calls: dict = {}
        self._sel = None

    # -------------------------------------------------------------- input coercion
    @staticmethod
    def _coerce_query(query, d: int) -> torch.Tensor:
        """(H_q, D), (1, H_q, 1, D) or, for B sequences, (B, H_q, 1, D) -> (B*H_q, D)
        (kernels/triton_search_wrappers.py:9-27)."""
        if not isinstance(query, torch.Tensor):
            raise TypeError(f"q must be a torch.Tensor, got {type(query)}")
        if query.ndim == 4:
            if query.shape[2] != 1:
                raise ValueError(f"4D query must be (B,H,1,D), got {tuple(query.shape)}")
            query = query.squeeze(2).reshape(-1, query.shape[-1])
        elif query.ndim != 2:
            raise ValueError(f"q must be (H,d) or (1,H,1,D), got {tuple(query.shape)}")
        if query.shape[-1] != d:
            raise ValueError(f"query dim mismatch: expected d={d}, got {query.shape[-1]}")
        return query

    @staticmethod
    def _coerce_threshold(t, h: int, device) -> torch.Tensor:
        """scalar or (H_q,) (kernels/triton_search_wrappers.py:57-71)."""
        if torch.is_tensor(t):
            t = t.to(device=device, dtype=torch.float32).reshape(-1)
        else:
            t = torch.tensor([float(t)], device=device, dtype=torch.float32)
        if t.numel() == 1 and h > 1:
            t = t.expand(h)
        if t.numel() != h:
            raise ValueError(f"threshold must be scalar or length H={h}, got {t.numel()}")
        return t.contiguous()

    @staticmethod
    def _coerce_scaling(scaling, h: int, device) -> torch.Tensor:
        """None or (H_q,) (kernels/triton_search_wrappers.py:74-89; the finiteness check
        there costs a host sync per call and is left to the caller)."""
        if scaling is None:
            return torch.ones((h,), device=device, dtype=torch.float32)
        if not torch.is_tensor(scaling):
            raise TypeError(f"scaling must be a torch.Tensor with shape (H,), got {type(scaling)}")
        s = scaling.to(device=device, dtype=torch.float32).reshape(-1)
        if s.numel() != h:
            raise ValueError(f"scaling must have length H={h}, got {s.numel()}")
        return s.contiguous()

    def _head_map(self, h_q: int, indexer, q_head_to_kv) -> Tuple[torch.Tensor, torch.Tensor, int, int]:
        """CSR of the query heads of each tree.  Default map: head h of sequence b belongs
        to tree b*H_kv + h // (H_q/H_kv) (searcher/cuda.py:23-33)."""
        t, batch, h_kv = indexer.num_trees, indexer.batch, indexer.num_heads
        key = (h_q, t, batch, None if q_head_to_kv is None
               else tuple(int(x) for x in torch.as_tensor(q_head_to_kv).reshape(-1).tolist()))
        hit = self._map_cache.get(key)
        if hit is not None:
            return hit
        if q_head_to_kv is None:
            if h_q % batch:
                raise ValueError(f"H_q={h_q} not divisible by batch={batch}")
            per_seq = h_q // batch
            if per_seq % h_kv:
                raise ValueError(
                    f"Unsupported head mapping: H_q={per_seq} must equal or be divisible "
                    f"by H_kv={h_kv}")
            # head h of the launch belongs to tree h // group: made on the device, nothing is copied there
            group = per_seq // h_kv
            val = (torch.arange(0, h_q + 1, group, dtype=torch.int32, device=indexer.device),
                   torch.arange(h_q, dtype=torch.int32, device=indexer.device), group, group)
            if not (val[0].is_cuda and torch.cuda.is_current_stream_capturing()):  # (its fill has not run yet)
                self._map_cache = {key: val}
            return val
        else:
            if not torch.is_tensor(q_head_to_kv):
                raise TypeError(
                    f"q_head_to_kv must be a torch.Tensor or None, got {type(q_head_to_kv)}")
            m = q_head_to_kv.detach().to("cpu", torch.long).reshape(-1)
            if m.numel() != h_q:
                raise ValueError(f"q_head_to_kv length mismatch: expected H_q={h_q}, got {m.numel()}")
            if bool(((m < 0) | (m >= t)).any()):
                raise ValueError(f"q_head_to_kv values must be in [0, {t - 1}]")
        order = torch.argsort(m, stable=True)
        counts = torch.bincount(m, minlength=t)
        off = torch.zeros(t + 1, dtype=torch.int32)
        off[1:] = counts.cumsum(0).to(torch.int32)
        dev = indexer.device
        val = (off.to(dev), order.to(torch.int32).to(dev), int(counts.max().item()), 0)
        self._map_cache = {key: val}
        return val

    def _query_struct(self, query, threshold, indexer, q_head_to_kv, scaling):
        dev = indexer.device
        q = _lib.in_chunks(self._coerce_query(query, indexer.dim).to(device=dev, dtype=indexer.dtype).contiguous())
        h_q = q.shape[0]
        tau = self._coerce_threshold(threshold, h_q, dev)
        sc = self._coerce_scaling(scaling, h_q, dev)
        off, heads, gmax, group = self._head_map(h_q, indexer, q_head_to_kv)
        qs = _lib.HiraQuery(h_q, q.data_ptr(), tau.data_ptr(), sc.data_ptr(), off.data_ptr(),
                            heads.data_ptr(), gmax, group)
        return qs, (q, tau, sc, off, heads)

    def _call(self, query, threshold, indexer, q_head_to_kv, scaling) -> Tuple[_Call, int, tuple]:
        """(call description with its query filled in, H_q, tensors to keep alive until the launch)."""
        tree = indexer.tree_struct()
        dim = indexer.dim
        if q_head_to_kv is None and isinstance(query, torch.Tensor) and \
                query.dtype is indexer.dtype and query.is_contiguous():
            shape = query.shape
            nd = len(shape)
            if shape[-1] == dim and (nd == 2 or (nd == 4 and shape[2] == 1)):
                h_q = query.numel() // dim
                key = (get_ident(), id(tree), h_q)
                c = self._calls.get(key)
                if c is None:
                    off, heads, gmax, group = self._head_map(h_q, indexer, None)
                    qs = _lib.HiraQuery(h_q, None, None, None, off.data_ptr(), heads.data_ptr(), gmax, group)
                    if len(self._calls) >= self._MAX_CALLS:
                        self._calls.clear()
                    c = self._calls[key] = _Call(tree, qs, indexer.keys_buf.get_device(), (off, heads))
                if query.get_device() == c.dev:
                    dev, qs = c.dev, c.query
                    if isinstance(threshold, torch.Tensor) and threshold.dtype is torch.float32 and \
                            threshold.numel() == h_q and threshold.get_device() == dev and \
                            threshold.is_contiguous():
                        tau = threshold
                    else:
                        tau = self._coerce_threshold(threshold, h_q, indexer.device)
                    one = None
                    if scaling is None:
                        one = c.ones or self._unit_scale(c, h_q)
                        sc = None if one else self._coerce_scaling(None, h_q, indexer.device)
                    elif isinstance(scaling, torch.Tensor) and scaling.dtype is torch.float32 and \
                            scaling.numel() == h_q and scaling.get_device() == dev and \
                            scaling.is_contiguous():
                        sc = scaling
                    else:
                        sc = self._coerce_scaling(scaling, h_q, indexer.device)
                    at = query.data_ptr()
                    if at % 16:
                        query = _lib.in_chunks(query)
                        at = query.data_ptr()
                    qs.q, qs.tau, qs.scaling = at, tau.data_ptr(), one or sc.data_ptr()
                    return c, h_q, (query, tau, sc)
        qs, keep = self._query_struct(query, threshold, indexer, q_head_to_kv, scaling)
        return (_Call(tree, qs, indexer.keys_buf.get_device(), keep), qs.num_q_heads, keep)

    @staticmethod
    def _unit_scale(c: _Call, h_q: int) -> Optional[int]:
        """Address of the library's scale of one per head, or None: more heads than it holds, or a
        capture is the first to ask on this device (then a tensor of the call's own is used)."""
        if c.dev < 0 or h_q > _lib.HIRA_UNIT_SCALE_HEADS or torch.cuda.is_current_stream_capturing():
            return None
        with torch.cuda.device(c.dev):
            c.ones = _lib.lib().hira_unit_scale()
        return c.ones

    def _get_workspace(self, nbytes: int, device) -> torch.Tensor:
        if self._workspace is None or self._workspace.numel() < nbytes or \
                not _on(self._workspace, device):
            # zero once: the arrival counters inside must start at zero and are left at
            # zero by every call
            self._workspace = torch.zeros(max(nbytes, 1), dtype=torch.uint8, device=device)
        return self._workspace

    def _prepare_output_buffer(self, h_q: int, n: int, device, fill: bool = True) -> torch.Tensor:
        """searcher/cuda.py:35-54.  fill=False: the search writes the fill value itself."""
        if self._tmp_out is None or not _on(self._tmp_out, device) or \
                tuple(self._tmp_out.shape) != (h_q, n):
            self._tmp_out = torch.full((h_q, n), self.output_fill_value, device=device,
                                       dtype=torch.float32)
        elif fill:
            self._tmp_out.fill_(self.output_fill_value)
        return self._tmp_out

    def _run(self, indexer, c: _Call, attn: bool, queue_rows: int = 0):
        lib = _lib.lib()
        ws_ptr, ws_bytes = None, 0
        queue_ref = c.queue_ref if queue_rows else None
        launch = self.launch  # (as it is now: callers may replace it, or change its fields)
        if c.launch is not launch:
            c.follow_launch(launch)
        if attn:
            rows, options = c.ws_for
            now = bytes(launch)
            if queue_rows > rows or options != now:  # (more rows in the queue may mean more partials)
                c.ws_for = queue_rows, now
                c.ws_bytes = lib.hira_search_workspace_bytes(c.tree_ref, c.query_ref, queue_ref, c.launch_ref)
                c.ws_at = _COUNTERS - lib.hira_search_counter_bytes(c.tree_ref, c.query_ref, c.launch_ref)
            ws_bytes, at = c.ws_bytes, c.ws_at
            ws = self._workspace
            if at < 0:  # more counters than are kept apart: a workspace of the call's own
                at = 0
                ws = torch.zeros(ws_bytes, dtype=torch.uint8, device=indexer.device)
            elif ws is None or ws.get_device() != c.dev or ws.numel() < at + ws_bytes:
                ws = self._get_workspace(at + ws_bytes, indexer.device)
            ws_ptr = ws.data_ptr() + at
        rc = lib.hira_search(c.tree_ref, c.query_ref, queue_ref, c.out_ref, c.launch_ref, ws_ptr,
                             ws_bytes, _lib.stream_of(c.dev))
        if rc:
            _lib.check(rc)

    # -------------------------------------------------------------- public API
    def search(self, query, threshold, indexer, q_head_to_kv: Optional[torch.Tensor] = None,
               scaling: Optional[torch.Tensor] = None, *, index_space: Optional[str] = None,
               stats: Optional[torch.Tensor] = None) -> torch.Tensor:
        if indexer.keys_buf is None:
            raise ValueError("Indexer is not built: missing children tensor.")
        space = index_space or self.index_space
        slots = space == "slot"
        tree, dense = indexer._tree_struct, self._tmp_out
        if slots and tree is not None and dense is not None and q_head_to_kv is None and stats is None:
            # a call like one before it on this tree: in one step, if its tensors are ready
            c = self._calls.get((get_ident(), id(tree), dense.shape[0]))
            if c is not None:
                if c.launch is not self.launch:
                    c.follow_launch(self.launch)
                rc = _lib.host().search(c.at or c.addresses(), c.launch_at, query, threshold, scaling, dense, self.output_fill_value,
                                        _lib.stream_of(c.dev))
                if rc is not None:
                    if rc:
                        _lib.check(rc)
                    return dense
        c, h_q, keep = self._call(query, threshold, indexer, q_head_to_kv, scaling)
        n = indexer.size[0] if slots else indexer.num_keys
        # in slot space the search fills what it does not select itself: one launch per call
        dense = self._tmp_out
        if not slots or dense is None or dense.shape != (h_q, n) or dense.get_device() != c.dev:
            dense = self._prepare_output_buffer(h_q, n, indexer.device, fill=not slots)
        out = c.out
        out.dense, out.dense_stride = dense.data_ptr(), n
        out.dense_by_position, out.dense_fill = (0, 1) if slots else (1, 0)
        out.dense_fill_value = self.output_fill_value
        out.sel_index = out.sel_score = out.sel_count = out.attn_out = None
        out.stats = None if stats is None else stats.data_ptr()
        self._run(indexer, c, False)
        del keep
        return dense

    def search_compact(self, query, threshold, indexer, q_head_to_kv=None, scaling=None, *,
                       capacity: Optional[int] = None, index_space: Optional[str] = None):
        """Compact result: (index (H_q, cap) int32, score (H_q, cap) fp32 raw q.k,
        count (H_q,) int32); entries of a head are unordered."""
        space = index_space or self.index_space
        c, h_q, keep = self._call(query, threshold, indexer, q_head_to_kv, scaling)
        cap = int(capacity or indexer.size[0])
        dev = indexer.device
        if self._sel is None or self._sel[0].shape != (h_q, cap) or not _on(self._sel[0], dev):
            self._sel = (torch.empty((h_q, cap), dtype=torch.int32, device=dev),
                         torch.empty((h_q, cap), dtype=torch.float32, device=dev),
                         torch.zeros((h_q,), dtype=torch.int32, device=dev))
        idx, score, count = self._sel
        count.zero_()
        out = c.out
        out.dense = out.attn_out = out.stats = None
        out.dense_fill = 0
        out.dense_by_position = 1 if space == "position" else 0
        out.sel_index, out.sel_score, out.sel_count = idx.data_ptr(), score.data_ptr(), count.data_ptr()
        out.sel_cap = cap
        self._run(indexer, c, False)
        del keep
        return idx, score, count

    def sparse_attention(self, index: torch.Tensor, score: torch.Tensor, count: torch.Tensor,
                         indexer, q_head_to_kv=None, scaling=None,
                         out: Optional[torch.Tensor] = None) -> torch.Tensor:
        """softmax(scaling * score) V over given lists (``search_compact`` in the slot index
        space, possibly edited), fp32: index (H_q, cap) int32 key slots, score (H_q, cap) fp32 raw
        q.k, count (H_q,) int32.  Returns (H_q, Dv) fp32; zeros where a list is empty."""
        if indexer.values_buf is None:
            raise ValueError("the index was built without values: nothing to attend to")
        if index.ndim != 2 or index.shape != score.shape or count.shape != (index.shape[0],):
            raise ValueError(f"lists must be (H_q, cap), (H_q, cap), (H_q,): got "
                             f"{tuple(index.shape)}, {tuple(score.shape)}, {tuple(count.shape)}")
        h_q, cap = index.shape
        dev = indexer.device
        index = index.to(device=dev, dtype=torch.int32).contiguous()
        score = score.to(device=dev, dtype=torch.float32).contiguous()
        count = count.to(device=dev, dtype=torch.int32).contiguous()
        sc = self._coerce_scaling(scaling, h_q, dev)
        off, heads, gmax, group = self._head_map(h_q, indexer, q_head_to_kv)
        qs = _lib.HiraQuery(h_q, None, None, sc.data_ptr(), off.data_ptr(), heads.data_ptr(),
                            gmax, group)
        if out is None:
            out = torch.empty((h_q, indexer.vdim), dtype=torch.float32, device=dev)
        elif _out_type(out, h_q * indexer.vdim, indexer.keys_buf.get_device()) != _lib.HIRA_F32:
            raise ValueError("sparse_attention writes float32")
        tree = indexer.tree_struct()
        stream = _lib.current_stream(dev)
        _lib.check(_lib.lib().hira_sparse_attention(
            C.byref(tree), C.byref(qs), index.data_ptr(), score.data_ptr(), count.data_ptr(),
            int(cap), out.data_ptr(), stream))
        return out

    def search_attention(self, query, threshold, indexer, q_head_to_kv=None, scaling=None, *,
                         queue_keys: Optional[torch.Tensor] = None,
                         queue_values: Optional[torch.Tensor] = None,
                         out: Optional[torch.Tensor] = None,
                         stats: Optional[torch.Tensor] = None) -> torch.Tensor:
        """Fused search + softmax(scaling * q.K_S^T) V_S over the selected keys and, when
        given, every queued key (T, m, D) / value (T, m, Dv).  Returns (H_q, Dv) fp32, or ``out``:
        contiguous, fp32 or bf16 (the fp32 sums are then rounded where they are written)."""
        if indexer.values_buf is None:
            raise ValueError("the index was built without values: nothing to attend to")
        c, h_q, keep = self._call(query, threshold, indexer, q_head_to_kv, scaling)
        if out is None:
            out = torch.empty((h_q, indexer.vdim), dtype=torch.float32, device=indexer.keys_buf.device)
            c.query.out_dtype = _lib.HIRA_F32
        else:
            c.query.out_dtype = _out_type(out, h_q * indexer.vdim, c.dev)
        so = c.out
        so.dense = so.sel_index = so.sel_score = so.sel_count = None
        so.dense_by_position = so.dense_fill = 0
        so.attn_out = out.data_ptr()
        so.stats = None if stats is None else stats.data_ptr()
        rows = 0
        if queue_keys is not None and queue_keys.shape[-2] > 0:
            qk = self._queue_rows(queue_keys, indexer, c.dev, indexer.dim)
            qv = self._queue_rows(queue_values, indexer, c.dev, indexer.vdim)
            rows = qk.numel() // (indexer.num_trees * indexer.dim)
            if qv.numel() != rows * indexer.num_trees * indexer.vdim:
                raise ValueError(f"queue: keys {tuple(queue_keys.shape)} and values "
                                 f"{tuple(queue_values.shape)} hold different numbers of rows")
            kp, vp = qk.data_ptr(), qv.data_ptr()
            if (kp | vp) % 16:
                qk, qv = _lib.in_chunks(qk), _lib.in_chunks(qv)
                kp, vp = qk.data_ptr(), qv.data_ptr()
            qu = c.queue
            qu.keys, qu.values, qu.len, qu.cap = kp, vp, rows, rows
            keep = keep + (qk, qv)
        self._run(indexer, c, True, rows)
        del keep
        return out

    @staticmethod
    def _queue_rows(x: torch.Tensor, indexer, dev: int, width: int) -> torch.Tensor:
        """Queued rows of all trees, contiguous, in the index's storage type and on its device."""
        if x.dtype is indexer.dtype and x.get_device() == dev and x.is_contiguous() and \
                x.numel() % (indexer.num_trees * width) == 0:
            return x
        x = x.reshape(indexer.num_trees, -1, width)
        return x.to(device=indexer.device, dtype=indexer.dtype).contiguous()

    def decode_plan(self, indexer, num_q_heads: int, scaling: float) -> "DecodePlan":
        """The plan for (this index, head count, one softmax scale for all heads), made on
        first use and kept: callers that come once per decode step and layer (the attention
        function) then pay one library call per step."""
        plans = self._decode_plans
        key = (id(indexer), int(num_q_heads), scaling if type(scaling) is float else float(scaling))
        plan = plans.get(key)
        if plan is None or plan.indexer is not indexer:  # (ids are reused once an index is gone)
            scale = torch.full((num_q_heads,), float(scaling), dtype=torch.float32,
                               device=indexer.device)
            plan = plans[key] = self.plan_attention(indexer, num_q_heads, scaling=scale)
        return plan

    def plan_attention(self, indexer, num_q_heads: int, scaling=None, q_head_to_kv=None,
                       stats: Optional[torch.Tensor] = None) -> "DecodePlan":
        """Pre-resolve everything that does not change between decode steps (head map,
        scaling, workspace) so that a step is one library call on ready device tensors."""
        return DecodePlan(self, indexer, num_q_heads, scaling, q_head_to_kv, stats)


class DecodePlan:
    """One fused search + attention call per ``run``: ``query`` (H_q, D) in the tree dtype,
    ``threshold`` (H_q,) fp32 and ``out`` (H_q, Dv) fp32 (or bf16: the fp32 sums are then rounded
    where they are written) must be contiguous device tensors that start at a multiple of 16 bytes, as torch allocates them."""

    def __init__(self, searcher: HIPSearcher, indexer, num_q_heads: int, scaling, q_head_to_kv,
                 stats):
        if indexer.values_buf is None:
            raise ValueError("the index was built without values: nothing to attend to")
        self.indexer = indexer
        self.searcher = searcher
        self.lib = _lib.lib()
        self._search_sampled = self.lib.hira_search_sampled
        dev = indexer.device
        self._dev = indexer.keys_buf.get_device()
        self.scaling = searcher._coerce_scaling(scaling, num_q_heads, dev)
        off, heads, gmax, group = searcher._head_map(num_q_heads, indexer, q_head_to_kv)
        self._keep = (off, heads, stats)
        self.query = _lib.HiraQuery(num_q_heads, None, None, self.scaling.data_ptr(),
                                    off.data_ptr(), heads.data_ptr(), gmax, group)
        self.out = _lib.HiraSearchOut()
        self.out.stats = None if stats is None else stats.data_ptr()
        self.launch = searcher.launch
        self.tree = indexer.tree_struct()
        self.queue = _lib.HiraQueue()
        self.sample = _lib.HiraSample()
        self._sample_ref = C.byref(self.sample)
        self.tau_buf: Optional[torch.Tensor] = None  # (H_q,) thresholds written by run_sampled
        self._ws_rows = 1  # queue rows the workspace is sized for
        self.ws_bytes = self._workspace_need()
        self.ws = torch.zeros(max(self.ws_bytes, 1), dtype=torch.uint8, device=dev)
        # (zero once: a launch that makes its thresholds hands them over in it and leaves it at zero)
        self.tau_scratch = torch.zeros((num_q_heads, 32), dtype=torch.float32, device=dev)
        self.sample.scratch = self.tau_scratch.data_ptr()
        self._refs = (C.byref(self.tree), C.byref(self.query), C.byref(self.out),
                      C.byref(self.launch), C.byref(self.queue))
        self._at: Optional[tuple] = None  # for ``attend``: the call's structs; where they lie, and the workspace

    def _workspace_need(self) -> int:
        fake_q = _lib.HiraQuery(self.query.num_q_heads, 1, 1, 1, 1, 1, self.query.max_group,
                                self.query.group_size)  # sizes only
        rows = _lib.HiraQueue(1, 1, self._ws_rows, self._ws_rows)
        return self.lib.hira_search_workspace_bytes(
            C.byref(self.tree), C.byref(fake_q), C.byref(rows), C.byref(self.launch))

    def _follow_index(self) -> None:
        """The index grew since the plan was made, or a queue holds more rows than before."""
        self.tree = self.indexer.tree_struct()
        need = self._workspace_need()
        if need > self.ws.numel():
            self.ws = torch.zeros(need, dtype=torch.uint8, device=self.indexer.device)
        self.ws_bytes = need
        self._refs = (C.byref(self.tree), C.byref(self.query), C.byref(self.out),
                      C.byref(self.launch), C.byref(self.queue))
        self._at = None

    def attend(self, query: torch.Tensor, samples: torch.Tensor, method: str, k: int, queue_keys: torch.Tensor,
               queue_values: torch.Tensor, rows: int) -> Optional[torch.Tensor]:
        """``run_sampled`` for the form that a running decode has, in one step: query (B, H_q, 1, D) of the tree's type, the
        first `rows` rows of a decode queue (B, H_kv, cap, D / Dv); makes the output (B, 1, H_q, Dv) in the query's type.
        None, and nothing done, for any other form, and where ``run_sampled`` is no longer this class's."""
        if getattr(self.run_sampled, "__func__", None) is not _RUN_SAMPLED:
            return None
        at = self._at
        if at is None or at[0] is not self.indexer._tree_struct:  # (moved, or not made since the index moved)
            if self.indexer._tree_struct is not self.tree:
                self._follow_index()
            structs = self.tree, self.query, self.sample, self.queue, self.out, self.launch
            at = self._at = *structs, (*map(C.addressof, structs), self._dev, self.ws, self.ws_bytes, self._ws_rows)
            if self.tau_buf is None:
                self.tau_buf = torch.empty((self.query.num_q_heads,), dtype=torch.float32, device=self.indexer.device)
        # (the structs stay alive with `at` while the call reads them, whoever replaces the plan's meanwhile)
        out = _lib.host().attend(at[6], self.tau_buf, query, samples, queue_keys, queue_values, rows,
                                 0 if method == "sample_max" else 1, k, _lib.stream_of(self._dev))
        if out.__class__ is int:
            _lib.check(out)
        return out

    def run(self, query: torch.Tensor, threshold: torch.Tensor, out: torch.Tensor,
            stream: Optional[int] = None, queue_keys: Optional[torch.Tensor] = None,
            queue_values: Optional[torch.Tensor] = None, queue_len: Optional[int] = None) -> None:
        """queue_keys / queue_values: (..., cap, D) / (..., cap, Dv) contiguous, tree dtype, the
        leading dimensions amounting to T trees: keys not in the index yet, attended by every
        head of their tree; the first `queue_len` rows of every tree are in use (all `cap`
        when not given)."""
        qu = self._step(query, out, queue_keys, queue_values, queue_len)
        self.query.tau = threshold.data_ptr()
        if stream is None:
            stream = _lib.stream_of(self._dev)
        t, q, o, l, _ = self._refs
        rc = self.lib.hira_search(t, q, qu, o, l, self.ws.data_ptr(), self.ws_bytes, stream)
        if rc:
            _lib.check(rc)

    def _step(self, query, out, queue_keys, queue_values, queue_len):
        """Query, output and queue of a step into the call's structs; the queue's reference, or None."""
        if self.indexer._tree_struct is not self.tree:  # (moved, or not made since the index moved)
            self._follow_index()
        q = self.query
        q.q = query.data_ptr()
        self.out.attn_out = out.data_ptr()
        kind = _OUT_TYPES.get(out.dtype)
        q.out_dtype = _refuse_out(out) if kind is None else kind
        if queue_keys is None or queue_len == 0:
            return None
        cap = queue_keys.shape[-2]
        if cap == 0:
            return None
        m = cap if queue_len is None else int(queue_len)
        if not 0 < m <= cap or queue_values.shape[-2] != cap:
            raise ValueError(f"queue: {m} rows in use of {cap} "
                             f"(values hold {queue_values.shape[-2]})")
        qs = self.queue
        qs.keys, qs.values, qs.len, qs.cap = queue_keys.data_ptr(), queue_values.data_ptr(), m, cap
        if m > self._ws_rows:
            # (a queue fills up row by row: not made anew for each of them, and no more than twice what the rows
            # in use take where they are few of the buffer's)
            self._ws_rows = min(cap, max(2 * m, 256))
            self._follow_index()
        return self._refs[4]

    def run_sampled(self, query: torch.Tensor, samples: torch.Tensor, method: str, k: int,
                    out: torch.Tensor, stream: Optional[int] = None,
                    queue_keys: Optional[torch.Tensor] = None,
                    queue_values: Optional[torch.Tensor] = None,
                    queue_len: Optional[int] = None, append=None) -> torch.Tensor:
        """A decode step whose thresholds come from a key sample (T, S, D), tree dtype,
        contiguous: ``hira_search_sampled`` ("sample_max" or "sample_mean_topk" with k) writes them
        into a buffer of the plan and searches with them, one or two launches of one call.  Returns that buffer.
        ``append`` = (new_keys (T, m, D), new_values (T, m, Dv) or None, state): the step first
        appends these rows to the index (``hira_update``'s arguments), in the launch that takes
        the thresholds (``hira_update_threshold``)."""
        tau = self.tau_buf
        if tau is None:
            tau = self.tau_buf = torch.empty((self.query.num_q_heads,), dtype=torch.float32,
                                             device=self.indexer.device)
        ix, shape = self.indexer, samples.shape
        if len(shape) != 3 or shape[0] != ix.num_trees or shape[2] != ix.dim or \
                samples.dtype is not ix.dtype or not samples.is_contiguous():
            raise ValueError(f"samples {tuple(shape)} {samples.dtype}: expected contiguous "
                             f"({ix.num_trees}, S, {ix.dim}) {ix.dtype}")
        if stream is None:
            stream = _lib.stream_of(self._dev)
        rule = 0 if method == "sample_max" else 1
        if append is not None:
            if self.indexer.tree_struct() is not self.tree:
                self._follow_index()
            self.query.q = query.data_ptr()
            new_keys, new_values, state = append
            rc = self.lib.hira_update_threshold(
                self._refs[0], new_keys.data_ptr(),
                new_values.data_ptr() if new_values is not None else None,
                int(new_keys.shape[-2]), state.data_ptr(), samples.data_ptr(),
                int(shape[1]), self._refs[1], rule, int(k), tau.data_ptr(), stream)
            if rc:
                _lib.check(rc)
            self.run(query, tau, out, stream, queue_keys, queue_values, queue_len)
            return tau
        qu = self._step(query, out, queue_keys, queue_values, queue_len)
        sm = self.sample
        sm.rows, sm.num_rows, sm.method, sm.k, sm.tau = samples.data_ptr(), shape[1], rule, int(k), tau.data_ptr()
        t, q, o, l, _ = self._refs
        rc = self._search_sampled(t, q, self._sample_ref, qu, o, l, self.ws.data_ptr(), self.ws_bytes, stream)
        if rc:
            _lib.check(rc)
        return tau


_RUN_SAMPLED = DecodePlan.run_sampled  # the one that ``attend`` stands for


class StreamingStep:
    """One decode step over a growing index as ONE captured HIP graph: append a key/value per
    tree (``hira_update``), thresholds from a key sample (optional; then ``hira_update_threshold``
    does both in one launch), search + sparse attention (``hira_search``) -- no host work between
    the launches and no read-back.  The graph works on fixed device buffers that ``step`` fills:
    ``new_keys`` (T, 1, D), ``new_values`` (T, 1, Dv), ``query`` (H_q, D), ``threshold`` (H_q)
    and writes ``out`` (H_q, Dv).  It is good for ``horizon`` steps (the index reserves room for
    that many appends and searches with level sizes fixed at their bound); ``refresh`` reads
    the sizes back and captures anew.  The reference does the same three things per decode
    token from Python with host synchronisation in between (cache/hira_cache.py:121-153,
    indexer/cuda.py:544-701)."""

    def __init__(self, searcher: HIPSearcher, indexer, num_q_heads: int, scaling=None, *,
                 horizon: int = 512, samples: Optional[torch.Tensor] = None,
                 method: str = "sample_mean_topk", k: int = 10, q_head_to_kv=None):
        if indexer.values_buf is None:
            raise ValueError("the index holds no values: nothing to attend to")
        self.searcher, self.indexer = searcher, indexer
        self.horizon = int(horizon)
        self.samples, self.method, self.k = samples, method, int(k)
        self._args = (num_q_heads, scaling, q_head_to_kv)
        dev, t = indexer.device, indexer.num_trees
        self.new_keys = torch.zeros((t, 1, indexer.dim), dtype=indexer.dtype, device=dev)
        self.new_values = torch.zeros((t, 1, indexer.vdim), dtype=indexer.dtype, device=dev)
        self.query = torch.zeros((num_q_heads, indexer.dim), dtype=indexer.dtype, device=dev)
        self.threshold = torch.zeros((num_q_heads,), dtype=torch.float32, device=dev)
        self.out = torch.zeros((num_q_heads, indexer.vdim), dtype=torch.float32, device=dev)
        self.refresh()

    def refresh(self) -> None:
        """Exact level sizes from the device, room for another ``horizon`` appends, new capture."""
        idx = self.indexer
        idx.begin_unsynced(self.horizon)
        h_q, scaling, q2kv = self._args
        self.plan = self.searcher.plan_attention(idx, h_q, scaling=scaling, q_head_to_kv=q2kv)
        lib, tree = _lib.lib(), idx.tree_struct()
        stream = torch.cuda.Stream(device=idx.device)
        stream.wait_stream(torch.cuda.current_stream(idx.device))
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(stream):
            with torch.cuda.graph(self.graph, stream=stream):
                if self.samples is not None:
                    # the append and the thresholds share a launch
                    self.plan.tau_buf = self.threshold
                    self.plan.run_sampled(self.query, self.samples, self.method, self.k, self.out,
                                          stream=stream.cuda_stream,
                                          append=(self.new_keys, self.new_values, idx._state))
                else:
                    _lib.check(lib.hira_update(C.byref(tree), self.new_keys.data_ptr(),
                                               self.new_values.data_ptr(), 1, idx._state.data_ptr(),
                                               stream.cuda_stream))
                    self.plan.run(self.query, self.threshold, self.out, stream=stream.cuda_stream)
        torch.cuda.current_stream(idx.device).wait_stream(stream)
        self.left = self.horizon

    def step(self, new_keys: torch.Tensor, new_values: torch.Tensor, query: torch.Tensor,
             threshold: Optional[torch.Tensor] = None) -> torch.Tensor:
        """new_keys / new_values: one row per tree (any shape with T*D / T*Dv elements), query
        (H_q, D); threshold (H_q,) unless the step takes it from the key sample.  Returns
        ``out`` (the graph's buffer: copy it before the next step if it has to survive)."""
        if self.left == 0:
            self.refresh()
        self.new_keys.copy_(new_keys.reshape(self.new_keys.shape))
        self.new_values.copy_(new_values.reshape(self.new_values.shape))
        self.query.copy_(query.reshape(self.query.shape))
        if self.samples is None:
            if threshold is None:
                raise ValueError("threshold missing (the step has no key sample to take it from)")
            self.threshold.copy_(threshold.reshape(self.threshold.shape))
        return self.replay()

    def replay(self) -> torch.Tensor:
        """The step on whatever the buffers hold (for callers that write new_keys, new_values,
        query and threshold in place, e.g. as outputs of their own kernels)."""
        if self.left == 0:
            self.refresh()
        self.graph.replay()
        self.indexer.note_unsynced(1)
        self.left -= 1
        return self.out


# the class name the reference's searcher/cuda.py defines (PyTorch-ROCm calls the device "cuda")
CUDASearcher = HIPSearcher
