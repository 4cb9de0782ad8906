"""The work that is timed when this framework's speed is judged: twelve listed cases, and `draw` for
more of the same ranges.  Every case goes through the public entry points as a serving program calls
them; sizes come from the repository's configurations, tests and benchmark, or are generic.

Kinds of case:

  decode    one decode step of one layer: `DecodePlan.run` over an index that the program keeps
            (range search + sparse attention of every query head), bf16
  attend    the same through the call without a plan, `HIPSearcher.search_attention`, with queued
            keys that the index does not hold yet; odd widths and fan-outs, fp32 and bf16
  search    `HIPSearcher.search`: the dense score matrix that the reference's searcher returns
  build     `HIPIndexer.build`: the index of a prompt
  append    an index over a short prompt that then takes windows of new keys (`HIPIndexer.update`
            with its read-back of the level sizes); the subtree rebuild of a long-running decode at
            its end where the tree has three levels
  generate  one request through the cache layer: `HiraCache.update` per layer for the prompt and for
            every token, `hira_attention_forward` for every token, thresholds from the key sample
            that the cache keeps (the prompt's own dense attention is torch's and not part of it)

Keys have a mean and a scale per channel, a query is a noisy copy of a key of its head, values are
standard normal; `massive` multiplies eight channels of keys and queries by 20.  The dense searches
run on clustered unit keys (256 clusters), which is what makes balls prune about as on a model's keys.
"""
import math
from types import SimpleNamespace

import torch

from hira_amd.attention.hira_attention import hira_attention_forward
from hira_amd.cache.hira_cache import HiraCache
from hira_amd.cache.hira_config import HiraConfig
from hira_amd.indexer import HIPIndexer
from hira_amd.searcher import HIPSearcher

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
DEV = "cuda"


def listed():
    return [
        # the shortest decode: a chat that has just begun (latency and launches count)
        dict(name="decode-2k", kind="decode", batch=1, h_kv=8, group=4, n=2000, d=128, dtype="bf16",
             levels=3, bf=32, frac=0.02, massive=False),
        # the headline configuration: 32k context, one sequence
        dict(name="decode-32k", kind="decode", batch=1, h_kv=8, group=4, n=32768, d=128, dtype="bf16",
             levels=3, bf=32, frac=0.01, massive=True),
        # batched serving: sixteen sequences of 32k
        dict(name="decode-16x32k", kind="decode", batch=16, h_kv=8, group=4, n=32768, d=128, dtype="bf16",
             levels=3, bf=32, frac=0.02, massive=True),
        # long context, eight query heads per KV head (the index then keeps its 8-bit shadow)
        dict(name="decode-128k-64h", kind="decode", batch=1, h_kv=8, group=8, n=131072, d=128, dtype="bf16",
             levels=4, bf=32, frac=0.01, massive=False),
        # fp32, a width and a fan-out that are no power of two, a ragged key count, a half-full queue
        dict(name="attend-5k-f32-odd", kind="attend", batch=1, h_kv=4, group=3, n=5003, d=80, dtype="f32",
             levels=4, bf=10, frac=0.02, queue=23),
        # the reference's published search shapes, smallest and largest: one fp32 head, ten keys kept
        dict(name="search-10k-f32", kind="search", heads=1, n=10000, d=128, dtype="f32", levels=3, bf=4),
        dict(name="search-90k-f32", kind="search", heads=1, n=90000, d=128, dtype="f32", levels=2, bf=8),
        # the index of a 32k prompt
        dict(name="build-32k", kind="build", h_kv=8, n=32768, d=128, dtype="bf16", levels=3, bf=32, iters=1,
             group=4),
        # the index of a 128k prompt (four levels, with the shadow)
        dict(name="build-128k", kind="build", h_kv=8, n=131072, d=128, dtype="bf16", levels=4, bf=32, iters=1,
             group=8),
        # a decode's keys folded into the index 64 tokens at a time, then one subtree re-clustered
        dict(name="append-64x24", kind="append", h_kv=8, n=8192, d=128, dtype="bf16", levels=3, bf=32,
             window=64, calls=24),
        # a request through the cache layer, as the integration guide configures it
        dict(name="generate-4k", kind="generate", layers=2, h_kv=8, group=4, n=4001, tokens=48, d=128,
             dtype="bf16", levels=3, bf=32, update_every=16),
        # the same with the configuration's defaults: five levels, fan-out 10, every token folded in at once
        dict(name="generate-1k-defaults", kind="generate", layers=2, h_kv=2, group=4, n=1111, tokens=24,
             d=64, dtype="bf16", levels=5, bf=10, update_every=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "attend", "search", "build", "append", "generate"])
    if kind == "decode":
        d, bf = rng.choice([64, 128, 128, 128, 256]), rng.choice([16, 32, 32, 64])
        batch, h_kv = rng.choice([1, 1, 2, 4, 16]), rng.choice([1, 2, 4, 8, 8])
        most = min(262144, 4194304 * 128 // (batch * h_kv * d))
        return dict(kind=kind, batch=batch, h_kv=h_kv, group=rng.choice([1, 3, 4, 4, 8]), n=_log(rng, 500, most),
                    d=d, dtype="bf16", levels=rng.choice([2, 3, 3, 4]), bf=bf,
                    frac=round(rng.uniform(0.005, 0.05), 4), massive=rng.random() < 0.5)
    if kind == "attend":
        return dict(kind=kind, batch=rng.choice([1, 2]), h_kv=rng.choice([1, 2, 4, 8]), group=rng.choice([1, 3, 4, 7]),
                    n=_log(rng, 300, 32768), d=rng.choice([32, 64, 80, 96, 128]), dtype=rng.choice(["f32", "bf16"]),
                    levels=rng.choice([2, 3, 4]), bf=rng.choice([4, 7, 10, 16, 24, 32]),
                    frac=round(rng.uniform(0.005, 0.05), 4), queue=rng.randrange(0, 65))
    if kind == "search":
        return dict(kind=kind, heads=rng.choice([1, 1, 2, 8]), n=_log(rng, 2000, 90000), d=rng.choice([64, 128, 128]),
                    dtype=rng.choice(["f32", "f32", "bf16"]), levels=rng.choice([2, 3]), bf=rng.choice([4, 8, 16, 32, 64]))
    if kind == "build":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
        bf, iters = rng.choice([16, 32, 32, 64]), rng.choice([1, 1, 2])
        # (fp32 keys are clustered on the vector units: shorter prompts; all rows meet all centres, so
        # the longest prompt goes with the root of the fan-out and of the rounds)
        most = min(131072, 131072 * math.sqrt(bf / 32 * 2 / (iters + 1))) if dtype == "bf16" else 20000
        return dict(kind=kind, h_kv=rng.choice([1, 2, 4, 8]), n=_log(rng, 500, most), d=rng.choice([64, 128, 128]),
                    dtype=dtype, levels=rng.choice([2, 3, 3, 4]), bf=bf, iters=iters, group=rng.choice([1, 4, 8]))
    if kind == "append":
        window = _log(rng, 1, 1024)
        return dict(kind=kind, h_kv=rng.choice([1, 2, 8]), n=_log(rng, 1000, 16384), d=rng.choice([64, 128]),
                    dtype=rng.choice(["bf16", "bf16", "f32"]), levels=rng.choice([2, 3, 3, 4]), bf=rng.choice([8, 16, 32]),
                    window=window, calls=max(2, min(32, 2048 // window)))
    levels, bf, every = rng.choice([(3, 32, 64), (3, 32, 16), (3, 16, 8), (5, 10, 1)])
    return dict(kind=kind, layers=rng.choice([1, 2]), h_kv=rng.choice([2, 4, 8]), group=rng.choice([1, 4, 8]),
                n=_log(rng, 300, 8000), tokens=rng.randrange(8, 49), d=rng.choice([64, 128]),
                dtype=rng.choice(["bf16", "bf16", "bf16", "f32"]), levels=levels, bf=bf, update_every=every)


# ------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _heads(g, batch, h_kv, d, massive):
    """Per sequence and KV head: mean and scale of every channel, eight channels boosted if massive."""
    mu, s = 0.3 * _randn(g, batch, h_kv, 1, d), torch.exp(0.5 * _randn(g, batch, h_kv, 1, d))
    boost = torch.ones((batch, h_kv, 1, d), device=DEV)
    if massive:
        pick = torch.rand((batch, h_kv, 1, d), generator=g, device=DEV).topk(8, dim=-1).indices
        boost.scatter_(-1, pick, 20.0)
    return mu, s, boost


def _keys(g, heads, n, dtype):
    mu, s, boost = heads
    batch, h_kv, _, d = mu.shape
    out = torch.empty((batch, h_kv, n, d), dtype=dtype, device=DEV)
    for b in range(batch):  # (a sequence at a time: the fp32 values are not kept)
        out[b] = ((mu[b] + s[b] * _randn(g, h_kv, n, d)) * boost[b]).to(dtype)
    return out


def _values(g, like):
    out = torch.empty_like(like)
    for b in range(like.shape[0]):
        out[b] = _randn(g, *like.shape[1:]).to(like.dtype)
    return out


def _queries(g, keys, heads, group):
    """(batch, h_kv * group, d): noisy copies of keys."""
    batch, h_kv, n, d = keys.shape
    j = torch.randint(0, n, (batch, h_kv, group, 1), generator=g, device=DEV)
    q = keys.gather(2, j.expand(-1, -1, -1, d)).float() + 0.5 * _randn(g, batch, h_kv, group, d) * heads[2]
    return q.reshape(batch, h_kv * group, d).to(keys.dtype)


def _taus(keys, q, count):
    """Thresholds halfway between the count-th and the next best score of every head."""
    batch, h_kv, n, d = keys.shape
    count, out = max(1, min(count, n - 1)), []
    for b in range(batch):
        qb = q[b].reshape(h_kv, -1, d).double()
        for h in range(h_kv):
            top = (keys[b, h].double() @ qb[h].t()).t().contiguous().topk(count + 1, dim=-1).values
            out.append(0.5 * (top[:, count - 1] + top[:, count]))
    return torch.cat(out).float().contiguous()


def prepare(case, seed):
    c = SimpleNamespace(**case)
    g, dtype = _gen(seed), DTYPES[c.dtype]
    s = SimpleNamespace(case=c)
    if c.kind in ("decode", "attend"):
        heads = _heads(g, c.batch, c.h_kv, c.d, getattr(c, "massive", False))
        keys = _keys(g, heads, c.n, dtype)
        values = _values(g, keys)
        h_q = c.batch * c.h_kv * c.group
        q = _queries(g, keys, heads, c.group)
        s.tau = _taus(keys, q, int(round(c.frac * c.n)))
        s.scale = torch.full((h_q,), c.d ** -0.5, device=DEV)
        s.index = HIPIndexer(c.levels, 1, c.bf, heads_per_tree=c.group).build(keys, values)
        s.searcher = HIPSearcher()
        if c.kind == "decode":
            s.q = q.reshape(h_q, c.d).contiguous()
            s.out = torch.empty((h_q, c.d), dtype=torch.float32, device=DEV)
            s.plan = s.searcher.plan_attention(s.index, h_q, scaling=s.scale)
        else:
            s.q = q.reshape(c.batch, c.h_kv * c.group, 1, c.d)
            s.qk = s.qv = None
            if c.queue:
                s.qk = _keys(g, heads, c.queue, dtype)
                s.qv = _values(g, s.qk)
    elif c.kind == "search":
        centres = _randn(g, 256, c.d)
        pick = torch.randint(0, 256, (c.heads, c.n), generator=g, device=DEV)
        keys = torch.nn.functional.normalize(centres[pick] + 0.15 * _randn(g, c.heads, c.n, c.d), dim=-1)
        keys = keys[None].to(dtype)
        s.q = torch.nn.functional.normalize(_randn(g, 1, c.heads, 1, c.d), dim=-1).to(dtype)
        s.tau = _taus(keys, s.q[:, :, 0], 10)
        s.index = HIPIndexer(c.levels, 1, c.bf).build(keys)
        s.searcher = HIPSearcher(block_c=c.bf)
    elif c.kind == "build":
        s.keys = _keys(g, _heads(g, 1, c.h_kv, c.d, False), c.n, dtype)
        s.values = _values(g, s.keys)
    elif c.kind == "append":
        heads = _heads(g, 1, c.h_kv, c.d, False)
        s.keys = _keys(g, heads, c.n, dtype)
        s.values = _values(g, s.keys)
        s.new = []
        for _ in range(c.calls):
            k = _keys(g, heads, c.window, dtype)
            s.new.append((k, _values(g, k)))
    else:
        s.model = SimpleNamespace(num_hidden_layers=c.layers, num_attention_heads=c.h_kv * c.group,
                                  num_key_value_heads=c.h_kv)
        s.model.get_text_config = lambda decoder=True: s.model
        s.config = HiraConfig(num_levels=c.levels, branching_factor=c.bf, update_every=c.update_every)
        s.module = SimpleNamespace(scaling=c.d ** -0.5)
        s.prompt, s.tokens = [], []
        for _ in range(c.layers):
            heads = _heads(g, 1, c.h_kv, c.d, False)
            keys = _keys(g, heads, c.n, dtype)
            s.prompt.append((keys, _values(g, keys)))
            k, q = _keys(g, heads, c.tokens, dtype), []
            for _ in range(c.tokens):
                q.append(_queries(g, keys, heads, c.group).reshape(1, c.h_kv * c.group, 1, c.d))
            v = _values(g, k)
            s.tokens.append([(k[:, :, t:t + 1].contiguous(), v[:, :, t:t + 1].contiguous(), q[t])
                             for t in range(c.tokens)])
    return s


# --------------------------------------------------------------------------------------------- runs
def _arrays(index):
    """The index as it stands: every array, the slots in use."""
    size = index.size
    out = {"perm": index.perm[:, : size[0]], "keys": index.keys_buf[:, : size[0]],
           "values": index.values_buf[:, : size[0]], "num_keys": index.num_keys}
    for l in range(1, index.num_levels):
        out["centers%d" % l] = index.centers[l][:, : size[l]]
        out["radii%d" % l] = index.radii[l][:, : size[l]]
        out["counts%d" % l] = index.counts[l][:, : size[l]]
    if index.q8:
        out["keys8"], out["kscale"] = index.keys8[:, : size[0]], index.kscale
        out["keps"] = index.keps[:, : size[1]]
    return out


def run(s):
    c = s.case
    if c.kind == "decode":
        s.plan.run(s.q, s.tau, s.out)
        return s.out
    if c.kind == "attend":
        return s.searcher.search_attention(s.q, s.tau, s.index, scaling=s.scale, queue_keys=s.qk,
                                           queue_values=s.qv)
    if c.kind == "search":
        return s.searcher.search(s.q, s.tau, s.index)
    if c.kind == "build":
        index = HIPIndexer(c.levels, c.iters, c.bf, heads_per_tree=c.group)
        return _arrays(index.build(s.keys, s.values))
    if c.kind == "append":
        index = HIPIndexer(c.levels, 1, c.bf).build(s.keys, s.values)
        for k, v in s.new:
            index.update(k, v)
        if c.levels >= 3 and not (index.tiled and c.bf % 16):
            index.rebuild_subtree(0)
        return _arrays(index)
    cache, outs = HiraCache(s.model, s.config), []
    for layer, (k, v) in enumerate(s.prompt):
        cache.update(k, v, layer)
    for t in range(c.tokens):
        for layer in range(c.layers):
            k, v, q = s.tokens[layer][t]
            held, _ = cache.update(k, v, layer)
            outs.append(hira_attention_forward(s.module, q, held, None, scaling=s.module.scaling)[0])
    return torch.cat(outs, dim=1)


# ------------------------------------------------------------------------------------- work, tolerance
def _build_work(trees, n, d, e, levels, bf, iters):
    """Keys and values read and written once, the centres written; the products of the nearest-centre
    passes that the clustering's definition has: every Lloyd round and the first packing round of a
    level, all rows against all centres."""
    nbytes, flops, rows = 4 * trees * n * d * e, 0, n
    for _ in range(1, levels):
        k = -(-rows // bf)
        flops += 2 * trees * rows * k * d * (iters + 1)
        nbytes += trees * k * (d * e + 8)
        rows = k
    return nbytes + 4 * trees * n, flops


def work(case):
    c = SimpleNamespace(**case)
    e = 4 if c.dtype == "f32" else 2
    if c.kind in ("decode", "attend"):
        # the keys read once (a threshold can fall anywhere), the selected values, queries, outputs
        trees = c.batch * c.h_kv
        union = min(1.0, c.frac * c.group)
        queue = getattr(c, "queue", 0)
        h_q = trees * c.group
        return {"bytes": trees * (c.n * c.d * e * (1 + union) + 2 * queue * c.d * e) + h_q * c.d * (e + 4),
                "flops": 2 * h_q * c.n * c.d * (1 + c.frac)}
    if c.kind == "search":
        return {"bytes": c.heads * c.n * (c.d * e + 4), "flops": 2 * c.heads * c.n * c.d}
    if c.kind == "build":
        b, f = _build_work(c.h_kv, c.n, c.d, e, c.levels, c.bf, c.iters)
        return {"bytes": b, "flops": f}
    if c.kind == "append":
        # every new row finds its node among the level-1 centres
        b, f = _build_work(c.h_kv, c.n, c.d, e, c.levels, c.bf, 1)
        new = c.window * c.calls
        return {"bytes": b + 4 * c.h_kv * new * c.d * e, "flops": f + 2 * c.h_kv * new * (c.n // c.bf) * c.d}
    b, f = _build_work(c.h_kv, c.n, c.d, e, c.levels, c.bf, 1)
    h_q = c.h_kv * c.group
    # per token and layer: the sample's rows for the thresholds, the keys of the search
    rows = min(1000, c.n) + c.n
    return {"bytes": c.layers * (b + c.tokens * (c.h_kv * rows * c.d * e + h_q * c.d * 2 * e)),
            "flops": c.layers * (f + c.tokens * 2 * h_q * rows * c.d)}


def tolerance(case):
    kind, f32 = case["kind"], case["dtype"] == "f32"
    if kind == "decode":
        # fp32 sums over exact bf16 products; logits reach thousands with the boosted channels, and
        # their rounding goes through exp()
        return {"rel": 2e-3 if case["massive"] else 1e-4}
    if kind == "attend":
        return {"rel": 3e-5 if f32 else 1e-4}
    if kind == "search":
        return {"rel": 1e-5}
    if kind in ("build", "append"):
        # the order of the keys is decided by fp32 comparisons: the same but for ties
        return {"rel": 1e-3, "max": 0.02, "differ": 0.001}
    return {"rel": 1e-4 if f32 else 1e-2}
