"""Performance cases of the paged KV path, each through its public entry points.

The path is what an attention layer and its runner call on paged KV caches: storing a chunk's or a step's K/V
(``store_kvcache``), a decode step's layers (``PagedKVDecodeAttention``: store, then paged decode attention), prefill
attention over pages (``paged_prefill_attention``) and in-place compaction of pruned contexts (``compact_kv_slots``).
The geometry is the repository's: 32 query heads over 8 KV heads (and its tensor-parallel shards), head_dim 128,
256-token pages scattered over a pool, E4M3FN payload with fp32 scales per token and KV head, or bf16 caches.
"""

from __future__ import annotations

import math
import random
import sys
from pathlib import Path
from types import SimpleNamespace

import torch

_PACKAGE = str(Path(__file__).resolve().parents[1] / "prism-infer_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

PAGE = 256
DIM = 128
FP8 = torch.float8_e4m3fn
SCALE = DIM ** -0.5
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def listed() -> list:
    return [
        # a prefill chunk of one layer enters the scaled FP8 cache
        {"name": "store_chunk_8192", "kind": "store", "tokens": 8192, "heads": 8, "input": "bf16", "cache": "scaled"},
        # a ragged prompt enters the unquantised cache (kv_cache_dtype auto)
        {"name": "store_dense_3001", "kind": "store", "tokens": 3001, "heads": 8, "input": "bf16", "cache": "bf16"},
        # the smallest call: one layer of one user's decode step, eager, an 8-image context of 1800 tokens
        {"name": "layer_b1_eager", "kind": "decode", "batch": 1, "min_len": 1800, "max_len": 1800, "q_heads": 32,
         "heads": 8, "cache": "scaled", "layers": 1, "graph": False, "sharers": 0, "shared": 0},
        # a few users' decode step replayed from a graph, as a server runs it (8 of the model's layers)
        {"name": "step_b4_graph", "kind": "decode", "batch": 4, "min_len": 700, "max_len": 4090, "q_heads": 32,
         "heads": 8, "cache": "scaled", "layers": 8, "graph": True, "sharers": 0, "shared": 0},
        # few users with long documents
        {"name": "step_b2_long_graph", "kind": "decode", "batch": 2, "min_len": 20000, "max_len": 32000, "q_heads": 32,
         "heads": 8, "cache": "scaled", "layers": 4, "graph": True, "sharers": 0, "shared": 0},
        # the batch of a loaded server: 64 mixed contexts, half of them behind one 4096-token system prefix
        {"name": "layers_b64_mixed", "kind": "decode", "batch": 64, "min_len": 1024, "max_len": 16380, "q_heads": 32,
         "heads": 8, "cache": "scaled", "layers": 4, "graph": False, "sharers": 32, "shared": 4096},
        # the same batch on one of eight tensor-parallel ranks
        {"name": "step_b64_tp8_graph", "kind": "decode", "batch": 64, "min_len": 1024, "max_len": 16380, "q_heads": 4,
         "heads": 1, "cache": "scaled", "layers": 4, "graph": True, "sharers": 32, "shared": 4096},
        # a batch over the unquantised cache
        {"name": "layers_b32_bf16", "kind": "decode", "batch": 32, "min_len": 300, "max_len": 4000, "q_heads": 32,
         "heads": 8, "cache": "bf16", "layers": 2, "graph": False, "sharers": 0, "shared": 0},
        # new prompts of mixed lengths in one prefill batch, nothing cached before them
        {"name": "prefill_prompts", "kind": "prefill", "batch": 6, "min_new": 61, "max_new": 1900, "prefix": 0,
         "q_heads": 32, "heads": 8, "input": "bf16"},
        # the largest: chunked prefill far into four long prompts
        {"name": "prefill_chunked", "kind": "prefill", "batch": 4, "min_new": 2048, "max_new": 2048, "prefix": 8192,
         "q_heads": 32, "heads": 8, "input": "bf16"},
        # a user's next message behind a long cached conversation
        {"name": "prefill_prefix_hit", "kind": "prefill", "batch": 2, "min_new": 90, "max_new": 240, "prefix": 12000,
         "q_heads": 32, "heads": 8, "input": "bf16"},
        # visual pruning after one multi-image prefill: every layer's kept slots move to the front, in place
        {"name": "compact_visual", "kind": "compact", "batch": 1, "tokens": 1800, "layers": 36, "heads": 8},
    ]


def _log_uniform(rng, low, high) -> int:
    return min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))


def draw(rng) -> dict:
    while True:
        kind = rng.choice(["store", "decode", "decode", "decode", "prefill", "prefill", "compact"])
        if kind == "store":
            return {"kind": kind, "tokens": _log_uniform(rng, 1, 8192), "heads": rng.choice([8, 8, 4, 1]),
                    "input": rng.choice(["bf16", "bf16", "f16"]), "cache": rng.choice(["scaled", "scaled", "bf16"])}
        if kind == "compact":
            return {"kind": kind, "batch": rng.randint(1, 4), "tokens": _log_uniform(rng, 300, 4000),
                    "layers": rng.randint(8, 36), "heads": rng.choice([8, 8, 4])}
        q_heads, heads = rng.choice([(32, 8), (32, 8), (16, 4), (8, 2), (4, 1)])
        if kind == "decode":
            batch = _log_uniform(rng, 1, 64)
            max_len = _log_uniform(rng, 256, 32000)
            min_len = max(1, int(max_len * rng.uniform(0.06, 1.0)))
            shared = rng.choice([0, 0, 256 * (min_len // 512)])
            case = {"kind": kind, "batch": batch, "min_len": min_len, "max_len": max_len, "q_heads": q_heads,
                    "heads": heads, "cache": rng.choice(["scaled", "scaled", "bf16"]), "layers": rng.randint(1, 4),
                    "graph": rng.random() < 0.5, "sharers": batch // 2 if shared and batch > 3 else 0,
                    "shared": shared if batch > 3 else 0}
            if work(case)["bytes"] <= 4e9:
                return case
        else:
            max_new = _log_uniform(rng, 16, 3000)
            case = {"kind": kind, "batch": rng.randint(1, 6), "min_new": max(1, int(max_new * rng.uniform(0.03, 1.0))),
                    "max_new": max_new, "prefix": rng.choice([0, _log_uniform(rng, 100, 12000)]), "q_heads": q_heads,
                    "heads": heads, "input": rng.choice(["bf16", "bf16", "f16"])}
            if work(case)["flops"] <= 1.2e12:
                return case


# ---------------------------------------------------------------- sizes that follow from the case alone

def _context_lens(case) -> list:
    r = random.Random(f"decode {case['batch']} {case['min_len']} {case['max_len']}")
    return [r.randint(case["min_len"], case["max_len"]) for _ in range(case["batch"])]


def _new_lens(case) -> list:
    r = random.Random(f"prefill {case['batch']} {case['min_new']} {case['max_new']}")
    return [r.randint(case["min_new"], case["max_new"]) for _ in range(case["batch"])]


def _kept_positions(case) -> list:
    """Per sequence: 64 text tokens, then about 70 % of the visual ones."""

    r = random.Random(f"compact {case['batch']} {case['tokens']}")
    return [[p for p in range(case["tokens"]) if p < 64 or r.random() < 0.7] for _ in range(case["batch"])]


def _sharing(case, lens) -> list:
    order = sorted(range(len(lens)), key=lambda b: -lens[b])
    return sorted(order[:case["sharers"]])


def _token_bytes(case) -> int:
    """K and V (and scales) of one cached token of one layer."""

    return 2 * case["heads"] * (DIM + 4 if case["cache"] == "scaled" else 2 * DIM)


def work(case) -> dict:
    if case["kind"] == "store":
        item = 4 if case["input"] == "f32" else 2
        return {"bytes": case["tokens"] * (2 * case["heads"] * DIM * item + _token_bytes(case) + 4), "flops": 0}
    if case["kind"] == "compact":
        kept = _kept_positions(case)
        moved = sum(1 for k in kept for i, p in enumerate(k) if i != p)
        per_slot = 2 * case["layers"] * case["heads"] * (DIM + 4)
        return {"bytes": 2 * moved * per_slot + 16 * sum(map(len, kept)), "flops": 0}
    if case["kind"] == "decode":
        lens = _context_lens(case)
        tokens = sum(lens) - max(0, case["sharers"] - 1) * case["shared"]
        # q and output, the step's K/V in bf16 and their stored rows
        rows = 4 * case["q_heads"] * DIM + 4 * case["heads"] * DIM + _token_bytes(case)
        tables = sum(math.ceil(n / PAGE) for n in lens) * 4 + 8 * len(lens)
        return {"bytes": case["layers"] * (tokens * _token_bytes(case) + len(lens) * rows + tables),
                "flops": case["layers"] * 4 * DIM * case["q_heads"] * sum(lens)}
    new = _new_lens(case)
    pairs = sum(n * case["prefix"] + n * (n + 1) // 2 for n in new)
    tokens = sum(new) + case["batch"] * case["prefix"]
    return {"bytes": tokens * 2 * case["heads"] * (DIM + 4) + 4 * sum(new) * case["q_heads"] * DIM,
            "flops": 4 * DIM * case["q_heads"] * pairs}


def tolerance(case):
    if case["kind"] in ("store", "compact"):
        return "exact"
    # bf16 and f16 outputs, and softmax weights that enter the second product in 16 bits: 64-bit results differ by
    # 1.6e-3 to 2.4e-3 (2-norm)
    return {"rel": 1e-2, "max": 0.1}


# ---------------------------------------------------------------- inputs, in plain torch

def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _generator(seed):
    g = torch.Generator(device=_device())
    g.manual_seed(seed)
    return g


def _normal(g, *shape, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=g, device=_device(), dtype=torch.float32).to(dtype)


def _quantise(x):
    """[..., dim] -> E4M3FN payload and one fp32 scale per row."""

    xf = x.float()
    scale = torch.clamp(xf.abs().amax(dim=-1) / torch.full((), 448.0, device=x.device), min=1e-6)
    return torch.clamp(xf / scale[..., None], -448.0, 448.0).to(FP8), scale


def _filled_pool(g, pages, heads, cache):
    """(k, v, k_scale, v_scale) of `pages` pages holding N(0, 1) tokens."""

    both = []
    for _ in range(2):
        if cache != "scaled":
            both.append((_normal(g, pages, PAGE, heads, DIM), None))
            continue
        payload = torch.empty(pages, PAGE, heads, DIM, dtype=FP8, device=_device())
        scale = torch.empty(pages, PAGE, heads, device=_device())
        for p in range(0, pages, 512):
            n = min(512, pages - p)
            payload[p:p + n], scale[p:p + n] = _quantise(_normal(g, n, PAGE, heads, DIM))
        both.append((payload, scale))
    (k, ks), (v, vs) = both
    return k, v, ks, vs


def _scattered_tables(seed, lens, sharing=(), shared=0):
    """Block tables over a pool a quarter larger than what the sequences hold."""

    prefix = shared // PAGE
    needs = [math.ceil(n / PAGE) - (prefix if b in sharing else 0) for b, n in enumerate(lens)]
    total = sum(needs) + prefix
    pool = total + total // 4 + 1
    free = list(range(pool))
    random.Random(seed).shuffle(free)
    head, at, tables = free[:prefix], prefix, []
    for b, need in enumerate(needs):
        tables.append((head if b in sharing else []) + free[at:at + need])
        at += need
    return tables, pool


def _decode_inputs(case, seed):
    lens = _context_lens(case)
    # room for the next step's token
    tables, pool = _scattered_tables(seed, [n + 1 for n in lens], set(_sharing(case, lens)), case["shared"])
    g = _generator(seed)
    layers = []
    for _ in range(case["layers"]):
        k, v, ks, vs = _filled_pool(g, pool, case["heads"], case["cache"])
        layers.append(SimpleNamespace(
            k=k, v=v, ks=ks, vs=vs, q=2 * _normal(g, case["batch"], case["q_heads"], DIM),
            new_k=_normal(g, case["batch"], case["heads"], DIM), new_v=_normal(g, case["batch"], case["heads"], DIM)))
    return lens, tables, layers


def _prefill_inputs(case, seed):
    new = _new_lens(case)
    lens = [n + case["prefix"] for n in new]
    tables, pool = _scattered_tables(seed, lens)
    g = _generator(seed)
    k, v, ks, vs = _filled_pool(g, pool, case["heads"], "scaled")
    q = 2 * _normal(g, sum(new), case["q_heads"], DIM, dtype=DTYPES[case["input"]])
    return new, lens, tables, SimpleNamespace(k=k, v=v, ks=ks, vs=vs, q=q)


def _store_inputs(case, seed):
    """N(0, 1) rows with 1 % outliers x 20 and a seeded permutation of the slots."""

    g = _generator(seed)
    rows = []
    for _ in range(2):
        x = _normal(g, case["tokens"], case["heads"], DIM, dtype=torch.float32)
        x = torch.where(torch.rand(x.shape, generator=g, device=x.device) < 0.01, 20 * x, x)
        rows.append(x.to(DTYPES[case["input"]]))
    pages = 2 * math.ceil(case["tokens"] / PAGE)
    slots = torch.randperm(pages * PAGE, generator=g, device=_device())[:case["tokens"]]
    return rows[0], rows[1], slots.to(torch.int32), pages


# ---------------------------------------------------------------- the calls

def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return state.run(state)


def _prepare_store(case, seed):
    key, value, slots, pages = _store_inputs(case, seed)
    shape = (pages, PAGE, case["heads"], DIM)
    scaled = case["cache"] == "scaled"
    caches = [torch.zeros(shape, dtype=FP8 if scaled else torch.bfloat16, device=key.device) for _ in range(2)]
    scales = [torch.zeros(shape[:-1], device=key.device) for _ in range(2)] if scaled else [None, None]
    return SimpleNamespace(run=_run_store, key=key, value=value, slots=slots, caches=caches, scales=scales)


def _run_store(s):
    from prism_infer.ops.kv_cache_store import store_kvcache

    store_kvcache(s.key, s.value, s.caches[0], s.caches[1], s.slots, s.scales[0], s.scales[1])
    return [*s.caches, *(x for x in s.scales if x is not None)]


def _prepare_decode(case, seed):
    from prism_infer.engine.decode_attention import PagedKVDecodeAttention, pack_decode_metadata

    lens, tables, layers = _decode_inputs(case, seed)
    # this step's metadata and the next one's: a server refills one buffer between steps
    steps = []
    for ahead in (0, 1, 0):
        ctx = [n + ahead for n in lens]
        slots = [t[(n - 1) // PAGE] * PAGE + (n - 1) % PAGE for t, n in zip(tables, ctx)]
        steps.append(pack_decode_metadata(slots, ctx, tables, device=_device()))
    meta = steps.pop()
    attention = []
    for x in layers:
        a = PagedKVDecodeAttention(case["q_heads"], case["heads"], DIM, SCALE)
        a.k_cache, a.v_cache, a.k_scale_cache, a.v_scale_cache = x.k, x.v, x.ks, x.vs
        attention.append(a)
    s = SimpleNamespace(run=_run_decode, layers=layers, attention=attention, steps=steps, meta=meta, turn=0, graph=None)
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _attend(s)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            s.outputs = _attend(s)
        s.graph = graph
    return s


def _attend(s):
    return [a(x.q, x.new_k, x.new_v, s.meta) for a, x in zip(s.attention, s.layers)]


def _run_decode(s):
    s.meta.copy_(s.steps[s.turn])
    s.turn ^= 1
    if s.graph is not None:
        s.graph.replay()
        outputs = s.outputs
    else:
        outputs = _attend(s)
    caches = [[x.k.view(torch.uint8), x.v.view(torch.uint8), x.ks, x.vs] if x.ks is not None
              else [x.k.view(torch.int16), x.v.view(torch.int16)] for x in s.layers]
    return {"attention": outputs, "caches": caches}


def _prepare_prefill(case, seed):
    new, lens, tables, x = _prefill_inputs(case, seed)
    width = max(map(len, tables))
    starts = [0]
    for n in new:
        starts.append(starts[-1] + n)
    x.context = SimpleNamespace(
        block_tables=torch.tensor([t + [-1] * (width - len(t)) for t in tables], dtype=torch.int32, device=_device()),
        context_lens=torch.tensor(lens, dtype=torch.int32, device=_device()),
        cu_seqlens_q=torch.tensor(starts, dtype=torch.int32, device=_device()))
    x.q_heads, x.heads, x.run = case["q_heads"], case["heads"], _run_prefill
    return x


def _run_prefill(s):
    from prism_infer.ops.paged_prefill import paged_prefill_attention

    return paged_prefill_attention(s.q, s.k, s.v, s.context, num_heads=s.q_heads, num_kv_heads=s.heads, scale=SCALE,
                                   k_scale_cache=s.ks, v_scale_cache=s.vs)


def _prepare_compact(case, seed):
    kept = _kept_positions(case)
    tables, pool = _scattered_tables(seed, [case["tokens"]] * case["batch"])
    src = [t[p // PAGE] * PAGE + p % PAGE for t, k in zip(tables, kept) for p in k]
    dst = [t[i // PAGE] * PAGE + i % PAGE for t, k in zip(tables, kept) for i in range(len(k))]
    g = _generator(seed)
    shape = (2, case["layers"], pool * PAGE, case["heads"])
    payload = torch.randint(0, 255, (*shape, DIM), generator=g, device=_device(), dtype=torch.uint8)
    return SimpleNamespace(
        run=_run_compact, payload=payload.view(FP8), scales=torch.rand(shape, generator=g, device=_device()) / 100,
        src=torch.tensor(src, dtype=torch.long, device=_device()),
        dst=torch.tensor(dst, dtype=torch.long, device=_device()))


def _run_compact(s):
    from prism_infer.ops.kv_compaction import compact_kv_slots

    compact_kv_slots(s.payload, s.src, s.dst)
    compact_kv_slots(s.scales, s.src, s.dst)
    return [s.payload.view(torch.uint8), s.scales.view(torch.int32)]


_PREPARE = {"store": _prepare_store, "decode": _prepare_decode, "prefill": _prepare_prefill,
            "compact": _prepare_compact}


# ---------------------------------------------------------------- the same in 64 bits

def exact(case, seed):
    if case["kind"] == "store":
        return _exact_store(case, seed)
    if case["kind"] == "decode":
        return _exact_decode(case, seed)
    if case["kind"] == "prefill":
        return _exact_prefill(case, seed)
    return None  # moved bytes


def _exact_store(case, seed):
    key, value, slots, pages = _store_inputs(case, seed)
    payloads, scales = [], []
    for x in (key, value):
        cache = torch.zeros(pages * PAGE, case["heads"], DIM, dtype=torch.float64, device=x.device)
        if case["cache"] == "scaled":
            payload, scale = _quantise(x)
            rows = torch.zeros(pages * PAGE, case["heads"], dtype=torch.float64, device=x.device)
            rows[slots.long()] = scale.double()
            scales.append(rows.view(pages, PAGE, -1))
            cache[slots.long()] = payload.double()
        else:
            cache[slots.long()] = x.to(torch.bfloat16).double()
        payloads.append(cache.view(pages, PAGE, case["heads"], DIM))
    return [*payloads, *scales]


def _sequence(payload, scale, table, n):
    """One sequence's cached K or V, dequantised: [heads, n, dim]."""

    pages = torch.tensor(table[:math.ceil(n / PAGE)], device=payload.device)
    rows = payload[pages].flatten(0, 1)[:n].double()
    if scale is not None:
        rows = rows * scale[pages].flatten(0, 1)[:n].double()[..., None]
    return rows.transpose(0, 1).contiguous()


def _attention(q, k, v, mask=None):
    """q [heads, rows, dim], k and v [heads, keys, dim] -> [heads, rows, dim]."""

    scores = torch.matmul(q, k.transpose(1, 2).contiguous()) * SCALE
    if mask is not None:
        scores.masked_fill_(~mask, -math.inf)
    return torch.matmul(torch.softmax(scores, dim=-1), v)


def _exact_decode(case, seed):
    lens, tables, layers = _decode_inputs(case, seed)
    group = case["q_heads"] // case["heads"]
    outputs = []
    for x in layers:
        stored = []
        for new, scaled in ((x.new_k, x.ks), (x.new_v, x.vs)):
            payload, scale = _quantise(new) if scaled is not None else (new, None)
            rows = payload.double() if scale is None else payload.double() * scale.double()[..., None]
            stored.append(rows)
        out = torch.empty(case["batch"], case["q_heads"], DIM, dtype=torch.float64, device=x.q.device)
        for b, (table, n) in enumerate(zip(tables, lens)):
            k, v = _sequence(x.k, x.ks, table, n), _sequence(x.v, x.vs, table, n)
            k[:, n - 1], v[:, n - 1] = stored[0][b], stored[1][b]
            out[b] = _attention(x.q[b].double().view(case["heads"], group, DIM), k, v).flatten(0, 1)
        outputs.append(out)
    return {"attention": outputs, "caches": [[None] * (4 if x.ks is not None else 2) for x in layers]}


def _exact_prefill(case, seed):
    new, lens, tables, x = _prefill_inputs(case, seed)
    group = case["q_heads"] // case["heads"]
    out = torch.empty(x.q.shape, dtype=torch.float64, device=x.q.device)
    at = 0
    for n, ctx, table in zip(new, lens, tables):
        k, v = _sequence(x.k, x.ks, table, ctx), _sequence(x.v, x.vs, table, ctx)
        visible = torch.arange(ctx, device=k.device)[None, :] <= torch.arange(ctx - n, ctx, device=k.device)[:, None]
        for h in range(case["q_heads"]):
            kv = slice(h // group, h // group + 1)
            out[at:at + n, h] = _attention(x.q[at:at + n, h].double()[None], k[kv], v[kv], visible)[0]
        at += n
    return out
