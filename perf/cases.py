"""The framework's work as a user's program has it done, over the sizes it meets in earnest.

The cases follow one generation with a budgeted cache: prompts are attended over the packed
ragged layout (prefill, whole or in chunks), every decode step appends and attends in each layer
(one request, or a static batch), every few hundred steps an audit scores, selects and compacts,
with the margin's gradients before it, the eviction queue drains between audits, and recalled
rows are put back. Shapes are the repository's benchmark configurations (Llama-3.2-1B: 16 layers,
8 KV heads, d64, G4; Llama-3.1-8B: 32 layers, 8 KV heads, d128, G4; the hybrid shape: 16 managed
layers, 4 KV heads, d256, G6) and ragged variants around them.

A case is a dict with a ``kind``; each kind has its own fields, inputs and outputs:

``attention``    one layer's ``packed_attention``: ``length`` queries a head onto ``cached`` +
                 ``length`` keys (``spread`` makes the cached lengths of the heads ragged)
``decode``       one decode step of ``layers`` layers: per layer ``_C.append`` and then attention
                 over the grown cache, or, ``deferred``, attention with the step's row pending
                 and one ``_C.append_layers`` for all layers
``batch_decode`` one layer of a static batch: ``batch_append``, then attention
``audit``        ``AuditStep.run`` (score, pool, select, compact); with ``drains`` in its lazy
                 form, followed by that many ``evict_prefix`` batches
``head_scores``  ``scoring.temporal_head_scores``, the per-head drop-in scorer
``margin``       the audit's margin: head logits, row margins, their hidden gradients, and every
                 layer's pre-projection gradient
``reinsert``     ``Reinserter.run``: recalled rows from pinned host memory into every layer
"""

import math
from types import SimpleNamespace

import numpy as np
import torch
import torch.nn.functional as F

from code_for_iclr27_amd import _C, attention, audit, reinsert, scoring, vjp
from code_for_iclr27_amd.scoring import LayerState

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
DEVICE = "cuda"


def listed():
    return [
        # a short prompt of the 1B shape, f16: the smallest prefill call, an odd length
        {"name": "prefill-1b-333-f16", "kind": "attention", "batch": 1, "kv_heads": 8, "groups": 4,
         "dim": 64, "length": 333, "cached": 0, "spread": 0, "dtype": "f16"},
        # a long prompt of the 8B shape in one call
        {"name": "prefill-8b-8192", "kind": "attention", "batch": 1, "kv_heads": 8, "groups": 4,
         "dim": 128, "length": 8192, "cached": 0, "spread": 0, "dtype": "bf16"},
        # a further chunk of a long prompt (or a new turn) onto a ragged, already evicted cache
        {"name": "prefill-hybrid-chunk", "kind": "attention", "batch": 1, "kv_heads": 4,
         "groups": 6, "dim": 256, "length": 1000, "cached": 4000, "spread": 900, "dtype": "bf16"},
        # a decode step as the model runs it, small model: 32 short calls in a row
        {"name": "decode-1b-step", "kind": "decode", "layers": 16, "kv_heads": 8, "groups": 4,
         "dim": 64, "keys": 1900, "spread": 300, "deferred": False},
        # a decode step of the 8B shape with the appends in one launch at its end
        {"name": "decode-8b-deferred", "kind": "decode", "layers": 32, "kv_heads": 8, "groups": 4,
         "dim": 128, "keys": 2250, "spread": 0, "deferred": True},
        # one layer of a static batch of eight requests
        {"name": "decode-8b-batch8", "kind": "batch_decode", "batch": 8, "kv_heads": 8,
         "groups": 4, "dim": 128, "keys": 1500, "spread": 750},
        # the audit of the 8B shape, every selected slot removed at once
        {"name": "audit-8b", "kind": "audit", "layers": 32, "kv_heads": 8, "groups": 4,
         "dim": 128, "keys": 2250, "spread": 0, "window": 250, "evict": 250, "drains": 0,
         "gradient": "abs_normal"},
        # the 1B shape as the controller drives it: a lazy audit on ragged heads, the queue
        # drained in batches of eight a head
        {"name": "audit-1b-lazy", "kind": "audit", "layers": 16, "kv_heads": 8, "groups": 4,
         "dim": 64, "keys": 1950, "spread": 300, "window": 250, "evict": 100, "drains": 3,
         "gradient": "abs_normal"},
        # the hybrid shape: wide heads, six query heads a KV head, a long window
        {"name": "audit-hybrid", "kind": "audit", "layers": 16, "kv_heads": 4, "groups": 6,
         "dim": 256, "keys": 9216, "spread": 0, "window": 512, "evict": 1024, "drains": 0,
         "gradient": "lognormal"},
        # one KV head through the drop-in operators, as a program that keeps the original host
        # code calls them (once for each layer and head)
        {"name": "head-scores-8b", "kind": "head_scores", "groups": 4, "dim": 128, "keys": 2250,
         "window": 250, "dtype": "bf16"},
        # the margin of a batch of eight rows at the 8B head and its gradients
        {"name": "margin-8b-batch8", "kind": "margin", "rows": 8, "vocab": 128256,
         "hidden": 4096, "layers": 32, "query_heads": 32, "dim": 128, "dtype": "bf16"},
        # recall on the long 8B cache: 512 rows for each layer and head from the host
        {"name": "reinsert-8b-long", "kind": "reinsert", "layers": 32, "kv_heads": 8, "dim": 128,
         "keys": 33792, "spread": 0, "recalled": 512},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["attention", "attention", "attention", "decode", "batch_decode", "audit",
                       "audit", "head_scores", "margin", "reinsert"])
    dim = rng.choice([64, 128, 128, 256])
    kv_heads, groups = {64: (8, 4), 128: (8, 4), 256: (4, 6)}[dim]
    if rng.random() < 0.3:
        groups = rng.choice([1, 2, 5, 7, 8])
    if kind == "attention":
        length = _log_uniform(rng, 2, 4096)
        cached = rng.choice([0, _log_uniform(rng, 1, 4096)])
        return {"kind": kind, "batch": 1 if length > 512 else rng.randint(1, 3),
                "kv_heads": kv_heads, "groups": min(groups, 6), "dim": dim, "length": length,
                "cached": cached, "spread": rng.randint(0, cached // 2),
                "dtype": rng.choice(["bf16", "bf16", "f16"])}
    if kind == "decode":
        deferred = rng.random() < 0.5
        return {"kind": kind, "layers": rng.randint(4, 32 if deferred else 16),
                "kv_heads": kv_heads, "groups": groups, "dim": dim,
                "keys": _log_uniform(rng, 60, 8000), "spread": rng.randint(0, 50),
                "deferred": deferred}
    if kind == "batch_decode":
        return {"kind": kind, "batch": rng.randint(2, 16), "kv_heads": kv_heads,
                "groups": groups, "dim": dim, "keys": _log_uniform(rng, 60, 3000),
                "spread": rng.randint(0, 900)}
    if kind == "audit":
        keys = _log_uniform(rng, 700, 6000)
        return {"kind": kind, "layers": rng.randint(2, 16), "kv_heads": kv_heads,
                "groups": min(groups, 6), "dim": dim, "keys": keys,
                "spread": rng.randint(0, keys // 4), "window": rng.randint(33, 300),
                "evict": rng.randint(40, keys // 6), "drains": rng.choice([0, 0, 2]),
                "gradient": rng.choice(["abs_normal", "lognormal"])}
    if kind == "head_scores":
        return {"kind": kind, "groups": groups, "dim": dim, "keys": _log_uniform(rng, 500, 33792),
                "window": rng.randint(33, 300), "dtype": rng.choice(["bf16", "bf16", "f16"])}
    if kind == "margin":
        return {"kind": kind, "rows": rng.randint(1, 8),
                "vocab": _log_uniform(rng, 8001, 128256), "hidden": rng.choice([2048, 3072, 4096]),
                "layers": rng.randint(4, 32), "query_heads": 32, "dim": rng.choice([64, 128]),
                "dtype": rng.choice(["bf16", "bf16", "f16", "f32"])}
    keys = _log_uniform(rng, 1000, 30000)
    return {"kind": kind, "layers": rng.randint(4, 32), "kv_heads": kv_heads, "dim": dim,
            "keys": min(keys, 10000) if dim == 256 else keys, "spread": rng.randint(0, 400),
            "recalled": rng.randint(3, 700)}


def _dtype(case):
    return {**DTYPES, "f32": torch.float32}[case.get("dtype", "bf16")]


def _ragged(count, keys, spread, index=0):
    """``count`` head lengths in [keys, keys + spread] (layer or request ``index``): part of the
    case's shape, the same for inputs of any seed."""
    rng = np.random.default_rng([count, keys, spread, index])
    return [int(v) for v in rng.integers(keys, keys + spread + 1, size=count)]


def _attention_lengths(case):
    """All rows of every (request, KV head) segment, the queries' own ones included."""
    segments = case["batch"] * case["kv_heads"]
    cached = _ragged(segments, max(0, case["cached"] - case["spread"]), case["spread"])
    return [c + case["length"] for c in cached]


def _metadata(lengths, length):
    """The packed layout as CacheMetadata carries it."""
    lengths = np.asarray(lengths, dtype=np.int64)
    cumulative = np.concatenate(([0], np.cumsum(lengths))).astype(np.int32)
    queries = np.arange(len(lengths) + 1, dtype=np.int32) * length
    return SimpleNamespace(cu_seqlens_k=torch.from_numpy(cumulative).to(DEVICE),
                           max_seqlen_k=int(lengths.max()),
                           decoding_cu_seqlens_q=torch.from_numpy(queries).to(DEVICE))


def _positions(lengths):
    return torch.cat([torch.arange(n, device=DEVICE, dtype=torch.float32) for n in lengths])


class _Normal:
    """Normal values on the device from one seed."""

    def __init__(self, seed):
        self.generator = torch.Generator(device=DEVICE)
        self.generator.manual_seed(seed)

    def __call__(self, *shape, dtype=torch.bfloat16):
        return torch.randn(shape, generator=self.generator, device=DEVICE,
                           dtype=torch.float32).to(dtype)


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return state.run(state)


def _prepare_attention(case, seed):
    normal, dtype = _Normal(seed), _dtype(case)
    lengths = _attention_lengths(case)
    heads = case["kv_heads"] * case["groups"]
    # as the query projection leaves them: [batch, length, heads, dim], seen head by head
    queries = normal(case["batch"], case["length"], heads, case["dim"], dtype=dtype).transpose(1, 2)
    return SimpleNamespace(
        run=_run_attention, queries=queries, keys=normal(sum(lengths), case["dim"], dtype=dtype),
        values=normal(sum(lengths), case["dim"], dtype=dtype), lengths=lengths,
        metadata=_metadata(lengths, case["length"]), length=case["length"],
        kv_heads=case["kv_heads"])


def _run_attention(s):
    return attention.packed_attention(s.queries, s.keys, s.values, s.metadata, s.length,
                                      s.kv_heads)


def _prepare_decode(case, seed):
    normal = _Normal(seed)
    heads, dim = case["kv_heads"], case["dim"]
    layers = []
    for layer in range(case["layers"]):
        lengths = _ragged(heads, case["keys"], case["spread"], layer)
        grown = [n + 1 for n in lengths]
        layers.append(SimpleNamespace(
            lengths=lengths, queries=normal(1, heads * case["groups"], 1, dim),
            keys=normal(sum(lengths), dim), values=normal(sum(lengths), dim),
            positions=_positions(lengths).reshape(-1, 1), new_keys=normal(1, heads, 1, dim),
            new_values=normal(1, heads, 1, dim), before=_metadata(lengths, 1),
            after=_metadata(grown, 1)))
    longest = max(max(layer.lengths) for layer in layers)
    return SimpleNamespace(run=_run_deferred if case["deferred"] else _run_decode, layers=layers,
                           heads=heads, logical=longest, maximum=longest + 1)


def _run_decode(s):
    results = []
    for layer in s.layers:
        keys, values, positions, _, _ = _C.append(
            layer.keys, layer.values, layer.positions, layer.new_keys, layer.new_values,
            layer.before.cu_seqlens_k, s.logical, s.maximum)
        out = attention.packed_attention(layer.queries, keys, values, layer.after, 1, s.heads)
        results.append((out, keys, values, positions))
    return results


def _run_deferred(s):
    outs = [attention.packed_attention(layer.queries, layer.keys, layer.values, layer.before, 1,
                                       s.heads, pending=(layer.new_keys, layer.new_values))
            for layer in s.layers]
    column = lambda name: [getattr(layer, name) for layer in s.layers]  # noqa: E731
    keys, values, positions, cumulative, lengths, _ = _C.append_layers(
        column("keys"), column("values"), column("positions"), column("new_keys"),
        column("new_values"), [layer.before.cu_seqlens_k for layer in s.layers],
        [s.logical] * len(s.layers), s.maximum)
    return {"out": outs, "cache": (keys, values, positions, cumulative, lengths)}


def _prepare_batch_decode(case, seed):
    normal = _Normal(seed)
    batch, heads, dim = case["batch"], case["kv_heads"], case["dim"]
    lengths = [_ragged(heads, case["keys"], case["spread"], request) for request in range(batch)]
    rows = [sum(row) for row in lengths]
    return SimpleNamespace(
        run=_run_batch_decode, lengths=lengths, heads=heads,
        keys=[normal(n, dim) for n in rows], values=[normal(n, dim) for n in rows],
        positions=[_positions(row).reshape(-1, 1) for row in lengths],
        new_keys=normal(batch, heads, 1, dim), new_values=normal(batch, heads, 1, dim),
        logical=[max(row) for row in lengths],
        queries=normal(batch, heads * case["groups"], 1, dim),
        after=_metadata([n + 1 for row in lengths for n in row], 1))


def _run_batch_decode(s):
    keys, values, positions = _C.batch_append(s.keys, s.values, s.positions, s.new_keys,
                                              s.new_values, s.lengths, s.logical)
    out = attention.packed_attention(s.queries, keys, values, s.after, 1, s.heads)
    return {"out": out, "cache": (keys, values, positions)}


def _prepare_audit(case, seed):
    normal = _Normal(seed)
    heads, groups, dim = case["kv_heads"], case["groups"], case["dim"]
    layers, longest = [], 0
    for layer in range(case["layers"]):
        lengths = _ragged(heads, case["keys"], case["spread"], layer)
        longest = max(longest, max(lengths))
        if case["gradient"] == "lognormal":
            gradient = torch.exp(1.5 * normal(heads * groups, dim, dtype=torch.float32))
        else:
            gradient = normal(heads * groups, dim, dtype=torch.float32).abs()
        layers.append(LayerState(normal(sum(lengths), dim), normal(sum(lengths), dim),
                                 _positions(lengths), lengths, None,
                                 normal(heads * groups, case["window"], dim), gradient))
    slots = case["layers"] * heads
    return SimpleNamespace(
        run=_run_audit, step=audit.AuditStep(), layers=layers,
        query_positions=torch.arange(longest - case["window"], longest, device=DEVICE),
        margin=torch.tensor([2.0], device=DEVICE), count=case["evict"] * slots,
        immediate=2 * slots if case["drains"] else None, drains=case["drains"], batch=8 * slots)


def _run_audit(s):
    outcome = s.step.run(s.layers, s.query_positions, s.margin, s.count, immediate=s.immediate)
    layers = outcome.layers
    for _ in range(s.drains):
        layers = outcome.queue.evict_prefix(layers, s.batch)
    return {"scores": outcome.scores, "pooled": outcome.pooled,
            "cache": (layers.keys, layers.values, layers.positions), "layout": layers.layout.block}


def _prepare_head_scores(case, seed):
    normal, dtype = _Normal(seed), _dtype(case)
    keys, window = case["keys"], case["window"]
    return SimpleNamespace(
        run=_run_head_scores, queries=normal(window, case["groups"], case["dim"], dtype=dtype),
        query_positions=torch.arange(keys - window, keys, device=DEVICE),
        keys=normal(keys, case["dim"], dtype=dtype), values=normal(keys, case["dim"], dtype=dtype),
        positions=_positions([keys]), last=keys - 32,
        gradient=normal(case["groups"], case["dim"], dtype=torch.float32).abs(),
        margin=torch.tensor([2.0], device=DEVICE))


def _run_head_scores(s):
    return scoring.temporal_head_scores(s.queries, s.query_positions, s.keys, s.positions,
                                        s.values, 0, s.last, s.gradient, s.margin, 1e-6, 64)


def _prepare_margin(case, seed):
    normal, dtype = _Normal(seed), _dtype(case)
    hidden, width = case["hidden"], case["query_heads"] * case["dim"]
    weight = normal(case["vocab"], hidden, dtype=dtype).mul_(hidden ** -0.5)
    embeddings = SimpleNamespace(weight=weight, bias=None)
    return SimpleNamespace(
        run=_run_margin, model=SimpleNamespace(get_output_embeddings=lambda: embeddings),
        weight=weight, hidden=normal(case["rows"], hidden, dtype=torch.float32).mul_(3.0),
        due=[float(r != 1) for r in range(case["rows"])], heads=case["query_heads"],
        dim=case["dim"],
        posts=[normal(hidden, dtype=torch.float32) for _ in range(case["layers"])],
        projections=[normal(hidden, width, dtype=dtype).mul_(width ** -0.5)
                     for _ in range(case["layers"])])


def _run_margin(s):
    logits = vjp.last_token_logits_float32(s.model, s.hidden)
    margins, targets, competitors = vjp.row_margins(logits)
    gradients = vjp.row_hidden_gradients(s.model, logits, targets, competitors, s.due)
    return {"logits": logits, "margins": margins, "targets": targets, "gradients": gradients,
            "pre": vjp.pre_gradients(s.posts, s.projections, s.heads, s.dim)}


def _prepare_reinsert(case, seed):
    normal = _Normal(seed)
    heads, dim, recalled = case["kv_heads"], case["dim"], case["recalled"]
    layers, identities = [], []
    for layer in range(case["layers"]):
        lengths = _ragged(heads, case["keys"], case["spread"], layer)
        positions = []
        for head, n in enumerate(lengths):
            # the head's positions: the resident ones and the recalled ones among them
            drawn = torch.randperm(n + recalled, generator=normal.generator, device=DEVICE)
            positions.append(drawn[recalled:].sort().values.float())
            identity = torch.empty((recalled, 3), dtype=torch.int64, device=DEVICE)
            identity[:, 0], identity[:, 1], identity[:, 2] = layer, head, drawn[:recalled]
            identities.append(identity)
        layers.append(LayerState(normal(sum(lengths), dim), normal(sum(lengths), dim),
                                 torch.cat(positions), lengths, None, None, None))
    metadata = torch.cat(identities)
    metadata = metadata[torch.randperm(len(metadata), generator=normal.generator, device=DEVICE)]
    payload = normal(len(metadata), 2, dim)
    return SimpleNamespace(run=_run_reinsert, reinserter=reinsert.Reinserter(), layers=layers,
                           payload=payload.cpu().pin_memory(),
                           metadata=metadata.cpu().pin_memory())


def _run_reinsert(s):
    merged = s.reinserter.run(s.layers, s.payload, s.metadata)
    return {"cache": (merged.layers.keys, merged.layers.values, merged.layers.positions),
            "rows": merged.recalled_rows, "layout": merged.layout.block}


def work(case):
    kind, size = case["kind"], 4 if case.get("dtype") == "f32" else 2
    dim, groups = case["dim"], case.get("groups", 0)
    if kind == "attention":
        length = case["length"]
        segments = case["batch"] * case["kv_heads"]
        cached = max(0, case["cached"] - case["spread"] / 2)
        pairs = segments * groups * length * (cached + (length + 1) / 2)
        return {"bytes": size * dim * segments * (2 * (cached + length) + 2 * groups * length),
                "flops": 4 * pairs * dim}
    if kind == "decode":
        segments = case["layers"] * case["kv_heads"]
        rows = segments * (case["keys"] + case["spread"] / 2)
        # each cached row read once, by the append or the attention, and written once
        return {"bytes": 2 * (rows + segments) * (2 * dim * 2 + 4) + 2 * segments * groups * dim * 2,
                "flops": 4 * groups * dim * (rows + segments)}
    if kind == "batch_decode":
        segments = case["batch"] * case["kv_heads"]
        rows = segments * (case["keys"] + case["spread"] / 2)
        return {"bytes": 2 * (rows + segments) * (2 * dim * 2 + 4) + 2 * segments * groups * dim * 2,
                "flops": 4 * groups * dim * (rows + segments)}
    if kind == "audit":
        slots = case["layers"] * case["kv_heads"]
        rows = slots * (case["keys"] + case["spread"] / 2)
        kept = rows - slots * (case["evict"] if not case["drains"] else 2)
        moved = sum(kept - 8 * slots * k for k in range(case["drains"] + 1))
        return {"bytes": rows * (2 * dim * 2 + 4) + slots * groups * (case["window"] * dim * 2 + dim * 4)
                + 8 * rows + moved * (2 * dim * 2 + 4) * (2 if case["drains"] else 1),
                "flops": 2 * rows * groups * case["window"] * dim + 2 * rows * groups * dim}
    if kind == "head_scores":
        return {"bytes": case["keys"] * (2 * dim * 2 + 8) + case["window"] * groups * dim * 2,
                "flops": 2 * case["keys"] * groups * dim * (case["window"] + 1)}
    if kind == "margin":
        head, rows = case["vocab"] * case["hidden"], case["rows"]
        width = case["query_heads"] * dim
        return {"bytes": 2 * head * size + rows * (case["vocab"] + 2 * case["hidden"]) * 4
                + case["layers"] * case["hidden"] * width * size,
                "flops": 4 * rows * head + 2 * case["layers"] * case["hidden"] * width}
    slots = case["layers"] * case["kv_heads"]
    resident = slots * (case["keys"] + case["spread"] / 2)
    recalled = slots * case["recalled"]
    return {"bytes": 2 * (resident + recalled) * (2 * dim * 2 + 4) + recalled * 24, "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("attention", "decode", "batch_decode"):
        # outputs rounded once to 16 bits: their own rounding is 1.7e-3 (bf16), 2.1e-4 (f16)
        # of the result, and another order of the f32 sums moves a few of them by one unit in
        # the last place (2^-8 or 2^-11 of the value)
        if case.get("dtype") == "f16":
            return {"rel": 8e-4, "max": 4e-3}
        return {"rel": 6e-3, "max": 3e-2}
    if kind == "audit":
        # scores are f32 from the same rounded logits (measured 2e-5 of the 64-bit ones at most);
        # the rows follow the selection, which stays the same apart from a cut between scores
        # that agree to the last bits
        return {"rel": 1e-4, "max": 2e-2, "differ": 1e-3}
    if kind == "head_scores":
        # as above: measured 3e-7 to 3.3e-6 of the 64-bit scores, of which a logit rounded to its
        # other 16-bit neighbour moves single ones further
        return {"rel": 1.5e-5, "max": 1e-2}
    if kind == "margin":
        return {"rel": 1e-5, "max": 1e-4, "differ": 1e-3}
    return "exact"


def _attend(queries, keys, values, lengths, length, kv_heads):
    """Causal grouped-query attention of every packed segment in 64 bits."""
    batch, heads, _, dim = queries.shape
    groups = heads // kv_heads
    out = torch.zeros((batch, length, heads, dim), dtype=torch.float64, device=keys.device)
    first = 0
    for index, n in enumerate(lengths):
        b, h = divmod(index, kv_heads)
        k, v = keys[first:first + n].double(), values[first:first + n].double()
        first += n
        for start in range(0, length, 1024):
            end = min(start + 1024, length)
            visible = (torch.arange(n, device=keys.device)[None, :]
                       <= torch.arange(start, end, device=keys.device)[:, None] + n - length)
            for g in range(groups):
                q = queries[b, h * groups + g, start:end].double()
                logits = (q @ k.T * dim ** -0.5).masked_fill(~visible, -torch.inf)
                out[b, start:end, h * groups + g] = torch.softmax(logits, -1) @ v
    return out.reshape(batch, length, heads * dim)


def _scores(queries, query_positions, keys, positions, values, first, last, gradient, margin,
            epsilon=1e-6):
    """One head's temporal scores in 64 bits, from logits that are rounded to the keys' type
    before and after the softmax scale, as the definition has them. ``queries`` [W, G, d]."""
    dtype = keys.dtype
    projected = gradient.double() @ values.double().T
    lowest, highest = None, None
    for start in range(0, queries.shape[0], 128):
        q = queries[start:start + 128]
        logits = (q.double() @ keys.double().T).to(dtype)
        logits = (logits.float() * (1.0 / math.sqrt(keys.shape[-1]))).to(dtype).double()
        hidden = positions.reshape(-1)[None, :] > query_positions[start:start + 128, None].float()
        p = torch.softmax(logits.masked_fill(hidden[:, None, :], -torch.inf), -1)
        outputs = (p * projected[None]).sum(-1, keepdim=True)
        drop = (p / (1.0 - p).clamp_min(epsilon) * (projected[None] - outputs)).sum(1)
        low, high = drop.amin(0)[first:last], drop.amax(0)[first:last]
        lowest = low if lowest is None else torch.minimum(lowest, low)
        highest = high if highest is None else torch.maximum(highest, high)
    margin = margin.double().reshape(())
    probability = torch.sigmoid(margin)

    def risk(d):
        return (probability * d - F.softplus(margin) + F.softplus(margin - d)).clamp_min(0.0)
    return torch.maximum(risk(lowest), risk(highest))


def exact(case, seed):
    kind, s = case["kind"], prepare(case, seed)
    if kind == "attention":
        return _attend(s.queries, s.keys, s.values, s.lengths, s.length, s.kv_heads)
    if kind == "decode":
        outs = []
        for layer in s.layers:
            keys, values = _appended(layer.keys, layer.values, layer.lengths,
                                     layer.new_keys, layer.new_values)
            outs.append(_attend(layer.queries, keys, values, [n + 1 for n in layer.lengths], 1,
                                s.heads))
        if case["deferred"]:
            return {"out": outs, "cache": None}
        return [(out, None, None, None) for out in outs]
    if kind == "batch_decode":
        lengths = [n for row in s.lengths for n in row]
        keys, values = _appended(torch.cat(s.keys), torch.cat(s.values), lengths, s.new_keys,
                                 s.new_values)
        return {"out": _attend(s.queries, keys, values, [n + 1 for n in lengths], 1, s.heads),
                "cache": None}
    if kind == "audit":
        scores, pooled = [], []
        for layer in s.layers:
            groups, first = layer.gradient.shape[0] // len(layer.head_lens), 0
            for head, n in enumerate(layer.head_lens):
                rows, query = slice(first, first + n), slice(head * groups, (head + 1) * groups)
                first += n
                scores.append(_scores(layer.queries[query].transpose(0, 1), s.query_positions,
                                      layer.keys[rows], layer.positions[rows],
                                      layer.values[rows], 0, n - 32, layer.gradient[query],
                                      s.margin))
                pooled.append(F.max_pool1d(scores[-1][None, None], 7, 1, 3).reshape(-1))
        return {"scores": torch.cat(scores), "pooled": torch.cat(pooled), "cache": None,
                "layout": None}
    if kind == "head_scores":
        return _scores(s.queries, s.query_positions, s.keys, s.positions, s.values, 0, s.last,
                       s.gradient, s.margin)
    if kind == "margin":
        logits, total = [], 0.0
        hidden = s.hidden.double()
        for start in range(0, case["vocab"], 8192):
            logits.append(hidden @ s.weight[start:start + 8192].double().T)
        logits = torch.cat(logits, 1)
        targets = logits.argmax(1)
        others = logits.scatter(1, targets[:, None], -torch.inf)
        margins = logits.gather(1, targets[:, None])[:, 0] - others.logsumexp(1)
        share = torch.softmax(others, 1)
        for start in range(0, case["vocab"], 8192):
            total = total + share[:, start:start + 8192] @ s.weight[start:start + 8192].double()
        due = torch.tensor(s.due, device=DEVICE, dtype=torch.float64)[:, None]
        pre = [(post.double() @ projection.double()).view(s.heads, s.dim)
               for post, projection in zip(s.posts, s.projections)]
        return {"logits": logits, "margins": margins, "targets": None,
                "gradients": (s.weight[targets].double() - total) * due, "pre": pre}
    return None


def _appended(keys, values, lengths, new_keys, new_values):
    """The packed rows with each segment's new row after its cached ones."""
    dim = keys.shape[1]
    parts = [torch.split(rows, lengths) for rows in (keys, values)]
    rows = [new.reshape(-1, dim) for new in (new_keys, new_values)]
    return tuple(torch.cat([x for i, part in enumerate(parts[t])
                            for x in (part, rows[t][i:i + 1])]) for t in (0, 1))
