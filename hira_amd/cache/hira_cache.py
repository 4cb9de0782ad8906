"""HiraCache / HiraCacheLayer: HuggingFace cache objects that own one index per layer.

Mirrors the reference's cache/hira_cache.py:19-249: the first ``update`` of a layer
(prefill) builds the index and returns the prefill tensors untouched; later updates queue
the new keys/values and fold the queue into the index every ``update_every`` tokens.
``update`` returns ``(CacheOutput, None)``, as the reference does, and the attention
function (attention/hira_attention.py) reads indexer, searcher and queue from it.

Both spellings of the two methods whose name or signature changed between transformers
releases are provided: ``get_max_cache_shape`` (reference, cache/hira_cache.py:167-168) /
``get_max_length``, and ``get_mask_sizes(cache_position tensor | query_length int)``.
"""
from __future__ import annotations

import ctypes as C
import inspect
from dataclasses import dataclass
from functools import lru_cache
from typing import Any

import torch
from transformers.cache_utils import Cache, CacheLayerMixin

from hira_amd import _lib
from hira_amd.cache.hira_config import DeviceMode, HiraConfig
from hira_amd.indexer import HIPIndexer
from hira_amd.searcher import HIPSearcher

# names the reference binds in this module (tests patch them there)
CUDAIndexer = HIPIndexer
CUDASearcher = HIPSearcher


@lru_cache(maxsize=64)
def _parameters(function) -> frozenset:
    """Names of a function's parameters (looked up once: the look costs as much as a token's launches)."""
    try:
        return frozenset(inspect.signature(function).parameters)
    except (TypeError, ValueError):
        return frozenset()


@dataclass
class CacheOutput:
    queued_keys: torch.Tensor
    queued_values: torch.Tensor
    prefill_keys: torch.Tensor | None
    prefill_values: torch.Tensor | None
    indexer: Any
    searcher: Any
    # beyond the reference's fields: the layer's key sample (B*H_kv, S, D) and the rule that
    # turns it into per-head thresholds (cache/hira_config.py:20-22 of the reference)
    samples: torch.Tensor | None = None
    threshold_method: str | None = None
    threshold_topk: int = 1
    # the buffers queued_keys / queued_values are views of: (B, H_kv, cap, D) in the index's
    # storage type and on its device, the first queued_keys.shape[-2] rows of every head in
    # use.  The attention function hands them to the library as they are.
    queue_store: tuple | None = None

    def __getattr__(self, name):
        # an output that a layer made knows how many rows of queue_store were in use; the two views
        # are taken when somebody looks at them (the attention function does not)
        rows = self.__dict__.get("queue_rows")
        if rows is not None and name in ("queued_keys", "queued_values"):
            view = self.queue_store[name == "queued_values"].narrow(2, 0, rows)
            self.__dict__[name] = view
            return view
        raise AttributeError(name)


class HiraCacheLayer(CacheLayerMixin):
    """One layer, all KV heads.  key_states / value_states: (B, H_kv, L, D)."""

    def __init__(
        self,
        device_mode: str,
        update_every: int,
        indexer_kwargs: dict[str, Any],
        searcher_kwargs: dict[str, Any],
        threshold_kwargs: dict[str, Any] | None = None,
    ):
        super().__init__()
        self.threshold_kwargs = threshold_kwargs or {}
        self.samples = None
        self.device_mode = device_mode
        self.update_every = update_every
        self.indexer_kwargs = indexer_kwargs
        self.searcher_kwargs = searcher_kwargs
        if self.device_mode == DeviceMode.CUDA_ONLY:
            # looked up at call time so that the module-level names can be replaced
            import hira_amd.cache.hira_cache as me

            self.indexer_cls = me.CUDAIndexer
            self.searcher_cls = me.CUDASearcher
        elif self.device_mode == DeviceMode.CPU_ONLY:
            raise NotImplementedError(
                "cpu_only is the reference's host path; this package is the MI355X path "
                "(device_mode='cuda_only')")
        else:
            raise NotImplementedError(f"Device mode {self.device_mode} not supported yet")
        self.indexed_len = 0
        self.queued_len = 0
        self._update_takes = None

    def _alloc_queue(self, rows: int):
        """Room for `rows` queued keys and values per head, allocated once (the reference
        concatenates per token, cache/hira_cache.py:121-140): in the index's storage type and
        on its device, so that a decode step passes the buffers on without a copy."""
        dt = getattr(self.indexer, "dtype", None) or self.dtype
        dev = getattr(self.indexer, "device", None) or self.device
        self._queue_k = torch.empty((self.batch, self.H_kv, rows, self.dim), dtype=dt, device=dev)
        self._queue_v = torch.empty((self.batch, self.H_kv, rows, self.vdim), dtype=dt, device=dev)
        self._queue_type = _lib.HIRA_F32 if dt == torch.float32 else _lib.HIRA_BF16
        esize = self._queue_k.element_size()
        if dt not in (torch.float32, torch.bfloat16) or self.dim * esize % 16 or self.vdim * esize % 16:
            self._queue_type = None
        # what a launch is told of the buffers beside where they lie, which is asked of the tensors each time: a
        # layer may be copied or pickled, and its copy's rows go into the copy's buffers
        self._queue_form = self._queue_type, self.batch * self.H_kv, rows
        self._queue_rows = rows
        self._queue_dev = self._queue_k.get_device()

    @property
    def queued_keys(self):
        return self._queue_k.narrow(2, 0, self.queued_len)

    @property
    def queued_values(self):
        return self._queue_v.narrow(2, 0, self.queued_len)

    def _whole_rows(self, x, m: int, width: int, like) -> bool:
        """Are x's rows (B, H_kv, m, width) -- or (H_kv, m, width) of one sequence --, one behind the
        other, on `like`'s device and 16-byte aligned, as the launches that copy rows take them?"""
        return (x.shape == (self.batch, self.H_kv, m, width) or (
            x.ndim >= 3 and x.shape[-3:] == (self.H_kv, m, width) and
            x.numel() == self.batch * self.H_kv * m * width)) and \
            x.get_device() == like.get_device() and x.is_contiguous() and x.data_ptr() % 16 == 0

    def _enqueue(self, key_states, value_states):
        n, dev = self.queued_len, self._queue_dev
        if dev >= 0 and n < self._queue_rows:
            # a token's rows, if they come as the queue holds them
            rc = _lib.host().enqueue(self._queue_k, self._queue_v, key_states, value_states, n, dev, _lib.stream_of(dev))
            if rc is not None:
                if rc:
                    _lib.check(rc)
                self.queued_len = n + 1
                return
        m = key_states.shape[-2]
        if self.queued_len + m > self._queue_k.shape[-2]:  # (a step of many tokens)
            old_k, old_v, n = self._queue_k, self._queue_v, self.queued_len
            self._alloc_queue(max(2 * old_k.shape[-2], n + m))
            self._queue_k[:, :, :n] = old_k[:, :, :n]
            self._queue_v[:, :, :n] = old_v[:, :, :n]
        k, v = self._queue_k, self._queue_v
        if self._queue_type is not None and self._queue_dev >= 0 and \
                key_states.dtype is k.dtype and value_states.dtype is k.dtype and \
                self._whole_rows(key_states, m, self.dim, k) and \
                self._whole_rows(value_states, m, self.vdim, v):
            # one launch for both
            rc = _lib.lib().hira_enqueue(
                k.data_ptr(), v.data_ptr(), *self._queue_form, self.queued_len, m, self.dim, self.vdim,
                key_states.data_ptr(), value_states.data_ptr(), _lib.stream_of(self._queue_dev))
            if rc:
                _lib.check(rc)
            self.queued_len += m
            return
        if key_states.ndim != 4:
            key_states = key_states.reshape(self.batch, self.H_kv, m, self.dim)
            value_states = value_states.reshape(self.batch, self.H_kv, m, self.vdim)
        self._queue_k.narrow(2, self.queued_len, m).copy_(key_states)
        self._queue_v.narrow(2, self.queued_len, m).copy_(value_states)
        self.queued_len += m

    def lazy_initialization(self, key_states, value_states):
        self.dim = key_states.shape[-1]
        self.vdim = value_states.shape[-1]
        self.H_kv = key_states.shape[-3]
        self.batch = key_states.shape[0] if key_states.ndim == 4 else 1
        self.dtype = key_states.dtype
        self.device = key_states.device
        self.indexer = self.indexer_cls(**self.indexer_kwargs)
        self.searcher = self.searcher_cls(**self.searcher_kwargs)
        self.queued_len = 0
        self._queue_k = self._queue_v = None  # allocated once the index knows its storage type
        self.keys = None  # the index holds the keys
        self.values = None
        self.is_initialized = True

    def update(self, key_states: torch.Tensor, value_states: torch.Tensor,
               cache_kwargs: dict[str, Any] | None = None, *args, **kwargs):
        if not self.is_initialized:
            self.lazy_initialization(key_states, value_states)
            self.indexer.build(key_states, value_states)
            # what the first append and the first subtree rebuild of a process load on first use
            # is loaded now, beside the prefill, not in the middle of the decode
            if hasattr(self.indexer, "warm_up"):
                try:
                    self.indexer.warm_up()
                except Exception as ex:  # (a courtesy, not a step of the prefill)
                    import warnings

                    warnings.warn(f"index warm-up skipped: {ex}")
            self._alloc_queue(max(1, min(int(self.update_every), 4096)))
            self.indexed_len = key_states.shape[-2]
            self._take_samples(key_states)
            self._sample_facts()
            return self._output(key_states, value_states), None
        if self.queued_len == 0 and key_states.shape[-2] >= self.update_every:
            # what would leave the queue at once does not pass through it
            if key_states.ndim != 4:
                key_states = key_states.reshape(self.batch, self.H_kv, -1, self.dim)
                value_states = value_states.reshape(self.batch, self.H_kv, -1, self.vdim)
            self._fold(key_states, value_states)
            return self._output(), None
        self._enqueue(key_states, value_states)
        if self.queued_len >= self.update_every:
            self.update_index()
        return self._output(), None

    def _take_samples(self, key_states):
        """A seeded random sample of the prompt's keys per KV head, for the sample-based
        threshold rules; none when the configured rule does not use one."""
        kw = self.threshold_kwargs
        if kw.get("method") not in ("sample_max", "sample_mean_topk") or kw.get("sample_size", 0) <= 0:
            return
        n = key_states.shape[-2]
        self._sample_target = min(int(kw["sample_size"]), 4096)
        s = min(self._sample_target, n)
        self._sample_gen = torch.Generator().manual_seed(12345)
        pick = torch.randperm(n, generator=self._sample_gen)[:s].sort().values
        k4 = key_states if key_states.ndim == 4 else key_states[None]
        # (in the index's storage dtype: the threshold kernel reads samples and queries alike)
        store = getattr(self.indexer, "dtype", None) or k4.dtype
        if k4.is_cuda and k4.dtype is store and self._queue_type is not None and \
                self._whole_rows(k4, n, self.dim, self._queue_k):
            # the positions travel with the launches: nothing waits for the build
            self.samples = torch.empty((k4.shape[0] * k4.shape[1], s, self.dim), dtype=store, device=k4.device)
            at = torch.arange(s, dtype=torch.int32), pick.to(torch.int32)
            self._replace_rows(self.samples, k4, n, n, *(C.cast(x.data_ptr(), C.POINTER(C.c_int32)) for x in at), s)
            return
        self.samples = k4[:, :, pick.to(k4.device)].reshape(-1, s, self.dim).to(store).contiguous()

    def _replace_rows(self, dst, src, rows: int, stride: int, slots, which, n: int):
        """dst[t][slots[i]] = src[t][which[i]] for every tree t and i < n (arrays of 32-bit numbers in host
        memory, read before the call returns); src holds `rows` rows a tree, `stride` rows apart."""
        _lib.check(_lib.lib().hira_replace_rows(
            dst.data_ptr(), self._queue_type, self.dim, dst.shape[0], dst.shape[1], src.data_ptr(), rows,
            stride, slots, which, n, _lib.stream_of(dst.get_device())))

    def _sample_pairs(self, new_keys, seen: int):
        """Keep the sample uniform over all indexed keys as the index grows (reservoir
        sampling, the same positions for every head): key number i (0-based) of the sequence
        joins with probability S/(i+1) in place of a random member; while the sample is still
        smaller than S every new key joins.  Returns the members to replace and the new keys that
        do, a member each at most."""
        if self.samples is None:
            return (), ()
        k4 = new_keys if new_keys.ndim == 4 else new_keys[None]
        m, first = k4.shape[-2], 0
        room = self._sample_target - self.samples.shape[1]
        if room > 0:  # a short prompt: the sample holds every key so far
            first = min(room, m)
            rows = k4.narrow(2, 0, first).reshape(-1, first, self.dim).to(self.samples.dtype)
            self.samples = torch.cat([self.samples, rows], dim=1).contiguous()
            self._sample_facts()
            if first == m:
                return (), ()
        s, seen = self.samples.shape[1], seen + first
        if self.samples.is_cuda:
            return _lib.host().draw(self._sample_gen, m - first, first, s, seen)
        # a layer in host memory (another indexer's) asks nothing of the library: the same numbers from torch
        draws = torch.rand(m - first, generator=self._sample_gen).tolist()
        who = [first + i for i, u in enumerate(draws) if u < s / (seen + i + 1)]
        if not who:
            return (), ()
        slots = torch.randint(0, s, (len(who),), generator=self._sample_gen).tolist()
        last = dict(zip(slots, who))  # (a slot drawn twice keeps its last arrival)
        return tuple(last.keys()), tuple(last.values())

    def _replace_sampled(self, new_keys, slots, which):
        """The members `slots` of the sample replaced by rows `which` of the new keys."""
        src = new_keys if new_keys.ndim == 4 else new_keys[None]
        m, smp = src.shape[-2], self.samples
        if smp.is_cuda and self._queue_type is not None:
            # one launch, the lists travel with its arguments.  (The rows of a head must lie one
            # behind the other and the heads evenly spaced, as the queue's and a model's do.)
            if src.dtype is not smp.dtype or src.get_device() != smp.get_device():
                src = src.to(device=smp.device, dtype=smp.dtype)
            b, h = src.shape[:2]
            step = src.stride(1) if h > 1 else src.stride(0) if b > 1 else m * self.dim
            if src.stride(3) != 1 or (m > 1 and src.stride(2) != self.dim) or \
                    step % self.dim or step < m * self.dim or (b > 1 and src.stride(0) != step * h) or \
                    src.data_ptr() % 16:
                # (clone: contiguous() would hand back a misaligned tensor as it is)
                src = src.clone(memory_format=torch.contiguous_format)
                step = m * self.dim
            arr = C.c_int32 * len(which)
            self._replace_rows(smp, src, m, step // self.dim, arr(*slots), arr(*which), len(which))
            return
        rows = src.reshape(-1, m, self.dim).to(smp.dtype)
        smp[:, torch.tensor(slots)] = rows[:, torch.tensor(which)].to(smp.device)

    def _sample_facts(self):
        """The rule as every output of the layer carries it."""
        kw = self.threshold_kwargs
        have = self.samples is not None
        self._rule = (kw.get("method") if have else None,
                      max(1, min(int(kw.get("topk", 1)), self.samples.shape[1] if have else 1)))

    def _output(self, prefill_keys=None, prefill_values=None):
        # (filled in directly: the views of the queue are taken when looked at)
        out = CacheOutput.__new__(CacheOutput)
        out.__dict__ = {
            "prefill_keys": prefill_keys, "prefill_values": prefill_values, "indexer": self.indexer,
            "searcher": self.searcher, "samples": self.samples, "threshold_method": self._rule[0],
            "threshold_topk": self._rule[1], "queue_store": (self._queue_k, self._queue_v),
            "queue_rows": self.queued_len}
        return out

    def update_index(self):
        self._fold(self.queued_keys, self.queued_values)
        self.queued_len = 0

    def _fold(self, keys, values):
        """New keys and values (B, H_kv, m, ...) into the index, and their share of the sample."""
        # no read-back of the level sizes: the host carries their bounds (HIPIndexer.update,
        # sync=False), so folding the queue into the index does not wait for the GPU; a
        # one-level index has no node counts to bound with and keeps the synchronous form
        if self._update_takes is None:
            update = self.indexer.update
            self._update_takes = _parameters(getattr(update, "__func__", update))
        kw = {}
        if "sync" in self._update_takes:  # (an indexer with the reference's update takes the rows alone)
            kw["sync"] = getattr(self.indexer, "num_levels", 1) < 2
        slots, which = self._sample_pairs(keys, self.indexed_len)
        if slots and "sample" in self._update_takes and self.samples.is_cuda and \
                self.samples.dtype is getattr(self.indexer, "dtype", None):
            # the sample's new members go with the append
            kw["sample"] = (self.samples, slots, which)
            slots = ()
        self.indexer.update(keys, values, **kw)
        if slots:
            self._replace_sampled(keys, slots, which)
        self.indexed_len += keys.shape[-2]

    def get_mask_sizes(self, cache_position):
        kv_offset = 0
        query_length = (int(cache_position) if isinstance(cache_position, int)
                        else cache_position.shape[0])
        return self.get_seq_length() + query_length, kv_offset

    def get_seq_length(self):
        if not self.is_initialized:
            return 0
        return self.indexed_len + self.queued_len

    def get_max_cache_shape(self):
        return -1

    def get_max_length(self):
        return -1

    def reset(self):
        if self.is_initialized:
            self.indexer = self.indexer_cls(**self.indexer_kwargs)
            self._queue_k = self._queue_v = None
            self.queued_len = 0
            self.indexed_len = 0
            self.samples = None
            self.is_initialized = False
        if hasattr(self, "cumulative_length"):
            self.cumulative_length = 0


class HiraCache(Cache):
    """HuggingFace ``Cache`` whose layers are HiraCacheLayer (cache/hira_cache.py:187-249)."""

    def __init__(self, cache_config, hira_config: HiraConfig):
        self.device_mode = hira_config.device_mode
        self.update_every = hira_config.update_every
        config = cache_config.get_text_config(decoder=True)
        layer_types = getattr(config, "layer_types", None)
        if layer_types is None:
            if getattr(config, "sliding_window", None) is not None:
                layer_types = ["sliding_attention" for _ in range(config.num_hidden_layers)]
            elif getattr(config, "attention_chunk_size", None) is not None:
                layer_types = ["chunked_attention" for _ in range(config.num_hidden_layers)]
            else:
                layer_types = ["full_attention" for _ in range(config.num_hidden_layers)]
        if hasattr(config, "num_kv_shared_layers"):
            layer_types = layer_types[: -config.num_kv_shared_layers]
        # query heads per KV head: the indexer's layout="auto" weighs it (an 8-bit shadow of the
        # keys pays from 8 heads a tree on)
        heads, kv_heads = (getattr(config, "num_attention_heads", None),
                           getattr(config, "num_key_value_heads", None))
        group = heads // kv_heads if heads and kv_heads and heads % kv_heads == 0 else None
        layers = [
            HiraCacheLayer(
                device_mode=self.device_mode,
                update_every=self.update_every,
                indexer_kwargs=self._indexer_kwargs(hira_config, group),
                searcher_kwargs=hira_config.get_searcher_kwargs(),
                threshold_kwargs=hira_config.get_threshold_kwargs(),
            )
            for _ in layer_types
        ]
        super().__init__(layers=layers, offloading=False)

    @staticmethod
    def _indexer_kwargs(hira_config: HiraConfig, group):
        """The configuration's indexer arguments, plus the heads per tree where the indexer in
        use takes them (one with the reference's constructor does not)."""
        import hira_amd.cache.hira_cache as me

        kw = dict(hira_config.get_indexer_kwargs())
        if group is not None and "heads_per_tree" in _parameters(me.CUDAIndexer.__init__):
            kw["heads_per_tree"] = group
        return kw

    def update(self, key_states: torch.Tensor, value_states: torch.Tensor, layer_idx: int,
               cache_kwargs: dict[str, Any] | None = None, *args, **kwargs):
        cache_output, _ = self.layers[layer_idx].update(key_states, value_states, cache_kwargs)
        return cache_output, None
