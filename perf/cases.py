"""The work that a serving program has this framework do, as cases to measure.

Each case is one call (or one fixed sequence of calls) through the package's
public entry points on GPU-resident inputs, as an engine makes them once per
layer or once per step:

* ``attention``: the registered ``"mi355x_paged"`` operator on one ragged batch
  (the step's K/V written into the paged cache, then attention over it);
* ``layer``: the fused steps of a decoder layer around the attention call
  (residual add + RMSNorm, q/k norm + rotary embedding + cache write, SwiGLU);
* ``edges``: the two ends of a decode step (greedy sampling of the logits, then
  the embedding and first norm of the sampled tokens);
* ``model``: a whole decode step of a small decoder, replayed from a HIP graph
  as the generation engine replays it, up to its logits.

A case's request lengths follow from its own fields (``shape_seed``), so its
work is the same for every seed; values and physical block ids come from the
seed.
"""

import math
import os
import random
import sys

import numpy as np
import torch

_PACKAGE_PARENT = os.path.join(os.getcwd(), "micro-vllm_amd")
if _PACKAGE_PARENT not in sys.path:
    sys.path.insert(0, _PACKAGE_PARENT)

from micro_vllm_amd import layers  # noqa: E402
from micro_vllm_amd.attention.attention import Attention  # noqa: E402
from micro_vllm_amd.attention.spec import ChunkedLocalSpec, FullAttentionSpec, SlidingWindowSpec  # noqa: E402

DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
EPS = 1e-6
ROPE_THETA = 500_000.0


def _attention(name, **fields):
    case = dict(
        kind="attention", dtype="bfloat16", q_heads=16, kv_heads=8, head_dim=128, block=16,
        decodes=0, context_lo=1, context_hi=1, chunks=0, chunk_lo=1, chunk_hi=1, prior_lo=0, prior_hi=0,
        spec="full", spec_size=0, hint=True, scale=1.0, shape_seed=0,
    )
    unknown = set(fields) - set(case)
    if unknown:
        raise ValueError(f"unknown fields {sorted(unknown)}")
    case.update(fields)
    return dict(case, name=name) if name else case


def listed():
    return [
        # A handful of short requests in float32, one of them still in its
        # prompt: the smallest call, and the dtype of the reference operator.
        _attention("small_mixed_f32", dtype="float32", decodes=3, context_lo=64, context_hi=255,
                   chunks=1, chunk_lo=17, chunk_hi=17),
        # Interactive serving: a few users decoding. An engine that builds its
        # metadata without the query-length hint.
        _attention("decode_8", decodes=8, context_lo=128, context_hi=4096, hint=False, scale=0.5),
        # A full decode batch with Qwen3-0.6B attention heads.
        _attention("decode_256", decodes=256, context_lo=128, context_hi=4096, scale=0.5),
        # Long documents with Llama-3-8B heads: the largest stream of K/V.
        _attention("decode_64_long", q_heads=32, decodes=64, context_lo=8192, context_hi=33280),
        # Continuous batching: prompt chunks beside running decodes.
        _attention("mixed_248_8x512", q_heads=32, decodes=248, context_lo=256, context_hi=8192,
                   chunks=8, chunk_lo=512, chunk_hi=512, prior_hi=2048),
        # The first step of a burst of fresh ragged prompts, in float16.
        _attention("prefill_prompts_f16", dtype="float16", chunks=16, chunk_lo=64, chunk_hi=1024, hint=False),
        # Chunked prefill deep inside long contexts: the most arithmetic.
        _attention("prefill_2x4096_long", q_heads=32, chunks=2, chunk_lo=4096, chunk_hi=4096,
                   prior_lo=4096, prior_hi=24576),
        # A sliding-window model with 32-token blocks, mixed step.
        _attention("window_mixed_f16", dtype="float16", q_heads=32, block=32, decodes=60, context_lo=256,
                   context_hi=8192, chunks=4, chunk_lo=300, chunk_hi=512, prior_hi=4096,
                   spec="window", spec_size=1024),
        # A model with 64-wide heads, mixed step of moderate size.
        _attention("dim64_mixed", q_heads=32, head_dim=64, decodes=30, context_lo=128, context_hi=2048,
                   chunks=2, chunk_lo=200, chunk_hi=256, prior_hi=512),
        # The fused layer steps of a full prefill step with Llama-3-8B sizes.
        dict(name="layer_8192", kind="layer", dtype="bfloat16", rows=8192, hidden=4096, q_heads=32, kv_heads=8,
             intermediate=14336, qk_norm=False, block=16),
        # Greedy sampling of a full decode batch and the next step's embedding.
        dict(name="edges_256", kind="edges", dtype="bfloat16", rows=256, vocab=151_936, hidden=1024),
        # A whole decode step: four layers of Qwen3-0.6B's shape and its head.
        dict(name="model_decode_256", kind="model", layers=4, decodes=256, context_lo=64, context_hi=1280,
             shape_seed=0),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case over the ranges that the listed ones stand for."""
    family = rng.choice(("decode", "decode", "mixed", "mixed", "prefill", "f32", "dim64", "layer", "edges", "model"))
    shape_seed = rng.randrange(1, 1 << 20)
    common = dict(
        dtype=rng.choice(("bfloat16", "bfloat16", "float16")), block=rng.choice((16, 16, 16, 32, 64)),
        hint=rng.random() < 0.5, scale=rng.choice((0.5, 1.0)), shape_seed=shape_seed,
    )
    kind = rng.choice(("full", "full", "full", "window", "chunked"))
    if kind != "full":
        common.update(spec=kind, spec_size=_log_int(rng, 48, 2048))
    if family == "decode":
        q_heads, kv_heads = rng.choice(((16, 8), (32, 8), (16, 8), (32, 8), (8, 8), (14, 2), (16, 1)))
        decodes = _log_int(rng, 1, 256)
        most = min(33_280, 5_200_000_000 // (decodes * kv_heads * 512))
        high = _log_int(rng, 64, max(64, most))
        return _attention(None, q_heads=q_heads, kv_heads=kv_heads, decodes=decodes,
                          context_lo=max(1, int(high * rng.uniform(0.02, 1.0))), context_hi=high, **common)
    if family in ("mixed", "prefill"):
        q_heads, kv_heads = rng.choice(((16, 8), (32, 8), (8, 8), (64, 8)))
        chunks = _log_int(rng, 1, 16)
        chunk_hi = _log_int(rng, 16, min(4096, 8192 // chunks))
        # At most the listed long prefill's arithmetic.
        most = int(1.8e12 / (4 * q_heads * 128 * chunks * chunk_hi)) - chunk_hi
        prior_hi = min(_log_int(rng, 16, 24_576), max(0, most))
        fields = dict(q_heads=q_heads, kv_heads=kv_heads, chunks=chunks,
                      chunk_lo=max(2, int(chunk_hi * rng.uniform(0.1, 1.0))), chunk_hi=chunk_hi, prior_hi=prior_hi)
        if family == "mixed":
            high = _log_int(rng, 64, 8192)
            fields.update(decodes=_log_int(rng, 1, 248), context_lo=max(1, int(high * rng.uniform(0.02, 1.0))),
                          context_hi=high)
        return _attention(None, **fields, **common)
    if family == "f32":
        common.update(dtype="float32", block=16)
        high = _log_int(rng, 16, 1024)
        return _attention(None, decodes=_log_int(rng, 1, 16), context_lo=max(1, high // 8), context_hi=high,
                          chunks=rng.randint(0, 2), chunk_lo=2, chunk_hi=_log_int(rng, 2, 64),
                          prior_hi=rng.choice((0, 200)), **common)
    if family == "dim64":
        high = _log_int(rng, 64, 2048)
        q_heads, kv_heads = rng.choice(((32, 8), (8, 2), (16, 8)))
        return _attention(None, head_dim=rng.choice((64, 64, 96)), q_heads=q_heads, kv_heads=kv_heads,
                          decodes=_log_int(rng, 1, 64), context_lo=max(1, high // 16), context_hi=high,
                          chunks=rng.randint(0, 2), chunk_lo=2, chunk_hi=_log_int(rng, 2, 256),
                          prior_hi=_log_int(rng, 1, 512), **common)
    if family == "layer":
        hidden, q_heads, inter, norm = rng.choice(((4096, 32, 14336, False), (1024, 16, 3072, True)))
        return dict(kind="layer", dtype=common["dtype"], rows=_log_int(rng, 1, 8192), hidden=hidden, q_heads=q_heads,
                    kv_heads=8, intermediate=inter, qk_norm=norm, block=16)
    if family == "edges":
        vocab, hidden = rng.choice(((151_936, 1024), (128_256, 4096)))
        return dict(kind="edges", dtype=common["dtype"], rows=_log_int(rng, 1, 256), vocab=vocab, hidden=hidden)
    return dict(kind="model", layers=rng.randint(1, 4), decodes=_log_int(rng, 1, 256), context_lo=64,
                context_hi=_log_int(rng, 128, 1280), shape_seed=shape_seed)


# ---- request shapes ---------------------------------------------------------------------


def _requests(case):
    """(context length, query count) of every request, from the case alone."""
    rng = random.Random(case["shape_seed"])
    chunk_lo, chunk_hi = case.get("chunk_lo", 1), case.get("chunk_hi", 1)
    got = []
    for _ in range(case.get("chunks", 0)):
        queries = rng.randint(chunk_lo, chunk_hi)
        got.append((rng.randint(case["prior_lo"], case["prior_hi"]) + queries, queries))
    for _ in range(case["decodes"]):
        got.append((rng.randint(case["context_lo"], case["context_hi"]), 1))
    return got


def _start(case, position):
    """First visible key of a query (an array of positions, or one)."""
    if case.get("spec", "full") == "window":
        return np.maximum(0, np.asarray(position) - case["spec_size"] + 1)
    if case.get("spec", "full") == "chunked":
        return np.asarray(position) // case["spec_size"] * case["spec_size"]
    return np.zeros_like(np.asarray(position))


def _keys_and_pairs(case):
    """Cache rows that some query of the batch sees, and visible (query, key) pairs."""
    keys = pairs = 0
    for length, queries in _requests(case):
        positions = np.arange(length - queries, length, dtype=np.int64)
        starts = _start(case, positions)
        keys += length - int(starts[0])
        pairs += int((positions - np.maximum(starts, starts[0]) + 1).sum())
    return keys, pairs


def _ragged(case, block, gen, device):
    """The batch's index tensors, its block ids drawn from a shuffled pool."""
    requests = _requests(case)
    counts = [-(-length // block) for length, _ in requests]
    pool = sum(counts) + sum(counts) // 20 + 16
    order = torch.randperm(pool, generator=gen, device=device)
    width = max(counts)
    table = torch.full((len(counts), width), pool, dtype=torch.int64, device=device)  # pads: the null block
    mask = torch.as_tensor(np.arange(width)[None, :] < np.asarray(counts)[:, None], device=device)
    table[mask] = order[: sum(counts)]
    positions = np.concatenate([np.arange(n - q, n, dtype=np.int64) for n, q in requests])
    owner = np.repeat(np.arange(len(requests)), [q for _, q in requests])
    pos = torch.as_tensor(positions, device=device)
    slots = table[torch.as_tensor(owner, device=device), pos // block] * block + pos % block
    return dict(
        positions=pos, table=table, slots=slots, pool=pool, width=width,
        qsl=torch.as_tensor(np.concatenate([[0], np.cumsum([q for _, q in requests])]).astype(np.int64), device=device),
        lengths=torch.as_tensor(np.asarray([n for n, _ in requests], dtype=np.int64), device=device),
        max_queries=max(q for _, q in requests),
    )


def _normal(shape, dtype, gen, device, scale=1.0):
    """N(0, 1) * scale, filled in pieces that bound the float32 temporaries."""
    out = torch.empty(shape, dtype=dtype, device=device)
    flat = out.view(-1)
    piece = 1 << 26
    for at in range(0, flat.numel(), piece):
        n = min(piece, flat.numel() - at)
        flat[at : at + n] = torch.randn(n, generator=gen, device=device) * scale
    return out


def _generator(seed, device):
    return torch.Generator(device=device).manual_seed(seed)


# ---- states and passes --------------------------------------------------------------------


def prepare(case, seed):
    device = torch.device("cuda", 0)
    gen = _generator(seed, device)
    return {"attention": _prepare_attention, "layer": _prepare_layer, "edges": _prepare_edges,
            "model": _prepare_model}[case["kind"]](case, gen, device, seed)


def run(state):
    return state["pass"](state)


def _prepare_attention(case, gen, device, seed):
    dtype, heads, dim, block = DTYPES[case["dtype"]], case["kv_heads"], case["head_dim"], case["block"]
    spec = {"full": lambda: FullAttentionSpec(), "window": lambda: SlidingWindowSpec(case["spec_size"]),
            "chunked": lambda: ChunkedLocalSpec(case["spec_size"])}[case["spec"]]()
    attention = Attention(spec, "mi355x_paged")
    r = _ragged(case, block, gen, device)
    tokens = r["positions"].numel()
    metadata = attention.build_metadata(
        query_positions=r["positions"], query_start_locations=r["qsl"], context_lengths=r["lengths"],
        block_table=r["table"], slot_mapping=r["slots"], block_size=block,
    )
    if case["hint"]:
        # Packing knows the largest query count without a device read.
        metadata = type(metadata)(
            query_positions=metadata.query_positions,
            query_context_start_positions=metadata.query_context_start_positions,
            query_start_locations=metadata.query_start_locations, context_lengths=metadata.context_lengths,
            block_table=metadata.block_table, slot_mapping=metadata.slot_mapping, block_size=block,
            max_query_len=r["max_queries"],
        )
    scale = case["scale"]
    return dict(
        {"pass": _run_attention}, attention=attention, metadata=metadata,
        query=_normal((tokens, case["q_heads"], dim), dtype, gen, device, scale),
        key=_normal((tokens, heads, dim), dtype, gen, device, scale),
        value=_normal((tokens, heads, dim), dtype, gen, device, scale),
        cache=_normal((2, r["pool"] + 1, block, heads, dim), dtype, gen, device, scale),
    )


def _run_attention(s):
    out = s["attention"](s["query"], s["key"], s["value"], s["cache"], s["metadata"])
    return {"out": out, "cache": s["cache"]}


def _rotary(positions, dim=128):
    inverse = 1.0 / (ROPE_THETA ** (torch.arange(0, dim, 2, dtype=torch.float32, device=positions.device) / dim))
    angles = torch.outer(positions.to(torch.float32), inverse)
    angles = torch.cat((angles, angles), dim=-1)
    return angles.cos().contiguous(), angles.sin().contiguous()


def _prepare_layer(case, gen, device, seed):
    dtype, rows, hidden = DTYPES[case["dtype"]], case["rows"], case["hidden"]
    q_heads, kv_heads, block = case["q_heads"], case["kv_heads"], case["block"]
    blocks = -(-rows // block) + 8
    positions = torch.randint(0, 4096, (rows,), generator=gen, device=device)
    cosine, sine = _rotary(torch.arange(4096, device=device))
    weight = lambda n: _normal((n,), dtype, gen, device, 0.1) + 1  # noqa: E731
    return dict(
        {"pass": _run_layer},
        x=_normal((rows, hidden), dtype, gen, device), residual=_normal((rows, hidden), dtype, gen, device, 4.0),
        norm=weight(hidden), qkv=_normal((rows, (q_heads + 2 * kv_heads) * 128), dtype, gen, device),
        gate_up=_normal((rows, 2 * case["intermediate"]), dtype, gen, device), q_heads=q_heads, kv_heads=kv_heads,
        q_norm=weight(128) if case["qk_norm"] else None, k_norm=weight(128) if case["qk_norm"] else None,
        cosine=cosine, sine=sine, positions=positions,
        cache=torch.zeros((2, blocks, block, kv_heads, 128), dtype=dtype, device=device),
        slots=torch.randperm(blocks * block, generator=gen, device=device)[:rows],
    )


def _run_layer(s):
    rows, nq, nkv = s["x"].shape[0], s["q_heads"] * 128, s["kv_heads"] * 128
    normed = layers.add_rms_norm(s["x"], s["norm"], EPS, s["residual"])
    q = s["qkv"][:, :nq].view(rows, -1, 128)
    k = s["qkv"][:, nq : nq + nkv].view(rows, -1, 128)
    v = s["qkv"][:, nq + nkv :].view(rows, -1, 128)
    rotated = layers.qk_norm_rope_kv_write(
        q, k, v, s["q_norm"], s["k_norm"], s["cosine"], s["sine"], EPS, s["cache"], s["slots"],
        positions=s["positions"],
    )
    activated = layers.silu_mul(s["gate_up"])
    return {"normed": normed, "residual": s["residual"], "query": rotated, "cache": s["cache"], "mlp": activated}


def _prepare_edges(case, gen, device, seed):
    dtype, vocab, hidden = DTYPES[case["dtype"]], case["vocab"], case["hidden"]
    return dict(
        {"pass": _run_edges}, logits=_normal((case["rows"], vocab), dtype, gen, device, 2.0),
        embedding=_normal((vocab, hidden), dtype, gen, device, 0.02),
        weight=_normal((hidden,), dtype, gen, device, 0.1) + 1,
    )


def _run_edges(s):
    tokens = layers.argmax_rows(s["logits"])
    residual, normed = layers.embed_rms_norm(tokens, s["embedding"], s["weight"], EPS)
    return {"tokens": tokens, "residual": residual, "normed": normed}


def _prepare_model(case, gen, device, seed):
    from micro_vllm_amd.attention.attention import AttentionMetadata
    from micro_vllm_amd.attention.operators.registry import get_attention_operator_class
    from micro_vllm_amd.harness.model import DecoderConfig, DecoderModel

    config = DecoderConfig.qwen3_0_6b(num_hidden_layers=case["layers"])
    operator = get_attention_operator_class("mi355x_paged")()
    model = DecoderModel(config, operator, device=device, seed=seed, fused_layers=True)
    model.build_rotary_table(1280)
    r = _ragged(case, 16, gen, device)
    metadata = AttentionMetadata(
        query_positions=r["positions"], query_context_start_positions=torch.zeros_like(r["positions"]),
        query_start_locations=r["qsl"], context_lengths=r["lengths"], block_table=r["table"],
        slot_mapping=r["slots"], block_size=16, max_query_len=1,
    )
    caches = [
        _normal((2, r["pool"] + 1, 16, config.num_key_value_heads, 128), torch.bfloat16, gen, device)
        for _ in range(case["layers"])
    ]
    ids = torch.randint(0, config.vocab_size, (case["decodes"],), generator=gen, device=device)
    state = dict({"pass": _run_model}, model=model, ids=ids, metadata=metadata, caches=caches)

    def step():
        return model.logits(model.forward(ids, r["positions"], caches, metadata))

    with torch.inference_mode():
        side = torch.cuda.Stream(device)
        side.wait_stream(torch.cuda.current_stream(device))
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream(device).wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state["logits"] = step()
    state["graph"] = graph
    return state


def _run_model(s):
    s["graph"].replay()
    return {"logits": s["logits"], "caches": s["caches"]}


# ---- what a pass cannot do without --------------------------------------------------------


def _attention_work(case, q_heads, kv_heads, dim, size):
    requests = _requests(case)
    tokens = sum(q for _, q in requests)
    keys, pairs = _keys_and_pairs(case)
    moved = (keys + 2 * tokens) * kv_heads * dim * 2 * size  # keys seen; new rows read and written
    moved += 2 * tokens * q_heads * dim * size
    moved += 8 * (sum(-(-n // case.get("block", 16)) for n, _ in requests) + 3 * tokens + 2 * len(requests) + 1)
    return moved, 4 * q_heads * dim * pairs


def work(case):
    if case["kind"] == "attention":
        size = 4 if case["dtype"] == "float32" else 2
        moved, flops = _attention_work(case, case["q_heads"], case["kv_heads"], case["head_dim"], size)
        return {"bytes": moved, "flops": flops}
    if case["kind"] == "layer":
        n, heads = case["rows"], case["q_heads"] + 2 * case["kv_heads"]
        moved = 2 * n * (4 * case["hidden"] + 2 * heads * 128 + 3 * case["intermediate"])
        moved += n * 16 + min(n, 4096) * 2 * 128 * 4
        return {"bytes": moved, "flops": n * (6 * case["hidden"] + 8 * 128 * heads + 6 * case["intermediate"])}
    if case["kind"] == "edges":
        n = case["rows"]
        return {"bytes": 2 * n * case["vocab"] + 2 * n * 3 * case["hidden"] + 16 * n,
                "flops": n * (case["vocab"] + 4 * case["hidden"])}
    n, hidden, inter, vocab = case["decodes"], 1024, 3072, 151_936
    weights = (32 * 128 + 16 * 128) * hidden + 3 * hidden * inter
    moved, flops = _attention_work(case, 16, 8, 128, 2)
    moved, flops = case["layers"] * (moved + 2 * weights), case["layers"] * (flops + 2 * n * weights)
    return {"bytes": moved + 2 * vocab * hidden + 2 * n * vocab, "flops": flops + 2 * n * vocab * hidden}


def tolerance(case):
    if case["kind"] == "attention":
        return {"float32": {"rel": 2e-6, "max": 1e-4}, "float16": {"rel": 2e-3, "max": 0.03},
                "bfloat16": {"rel": 1.2e-2, "max": 0.2}}[case["dtype"]]
    if case["kind"] == "model":
        return {"rel": 3e-2, "max": 0.3}
    # One 16-bit rounding of another value next to a rounding boundary, per
    # element; argmax indices are whole numbers and have to be the same.
    return {"rel": 1e-3, "max": 0.02, "differ": 0.0} if case["dtype"] == "bfloat16" else \
        {"rel": 2e-4, "max": 0.004, "differ": 0.0}


# ---- the same in 64 bits ------------------------------------------------------------------


def _exact_attention(case, q, k_new, v_new, cache, table, slots, lengths, q_heads, kv_heads, dim):
    """Attention output in float64 over the cache with the step's rows written."""
    block = case.get("block", 16)
    group = q_heads // kv_heads
    flat = cache.view(2, -1, kv_heads, dim).clone()
    flat[0, slots] = k_new.to(flat.dtype)
    flat[1, slots] = v_new.to(flat.dtype)
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    at = 0
    for r, (length, queries) in enumerate(_requests(case)):
        positions = np.arange(length - queries, length, dtype=np.int64)
        starts = np.maximum(_start(case, positions), _start(case, positions[:1]))
        first = int(starts[0])
        seen = torch.arange(first, length, device=q.device)
        rows = table[r, seen // block] * block + seen % block
        keys, values = flat[0, rows].double(), flat[1, rows].double()
        hidden = (seen[None, :] > torch.as_tensor(positions, device=q.device)[:, None]) | (
            seen[None, :] < torch.as_tensor(starts, device=q.device)[:, None])
        for h in range(kv_heads):
            queries_h = q[at : at + queries, h * group : (h + 1) * group].double()
            kt, vh = keys[:, h].t().contiguous(), values[:, h].contiguous()
            if queries == 1:
                scores = queries_h[0].contiguous() @ kt / math.sqrt(dim)
                out[at, h * group : (h + 1) * group] = torch.softmax(scores, dim=-1) @ vh
                continue
            for g in range(group):
                scores = queries_h[:, g].contiguous() @ kt / math.sqrt(dim)
                scores.masked_fill_(hidden, -math.inf)
                out[at : at + queries, h * group + g] = torch.softmax(scores, dim=-1) @ vh
        at += queries
    return out


def _exact_norm(x, weight):
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + EPS) * weight.double()


def _exact_rotate(x, cosine, sine):
    first, second = x.chunk(2, dim=-1)
    return x * cosine + torch.cat((-second, first), dim=-1) * sine


def exact(case, seed):
    with torch.inference_mode():
        s = prepare(case, seed)
        if case["kind"] == "attention":
            m = s["metadata"]
            out = _exact_attention(case, s["query"], s["key"], s["value"], s["cache"], m.block_table, m.slot_mapping,
                                   m.context_lengths, case["q_heads"], case["kv_heads"], case["head_dim"])
            return {"out": out, "cache": None}  # the cache holds copied bytes
        if case["kind"] == "layer":
            rows, nq, nkv = case["rows"], case["q_heads"] * 128, case["kv_heads"] * 128
            summed = s["x"].double() + s["residual"].double()
            qkv = s["qkv"].double()
            q, k = qkv[:, :nq].reshape(rows, -1, 128), qkv[:, nq : nq + nkv].reshape(rows, -1, 128)
            if case["qk_norm"]:
                q, k = _exact_norm(q, s["q_norm"]), _exact_norm(k, s["k_norm"])
            c, sn = (t[s["positions"]].double()[:, None] for t in (s["cosine"], s["sine"]))
            cache = s["cache"].double()
            flat = cache.view(2, -1, case["kv_heads"], 128)
            flat[0, s["slots"]] = _exact_rotate(k, c, sn)
            flat[1, s["slots"]] = qkv[:, nq + nkv :].reshape(rows, -1, 128)
            gate, up = s["gate_up"].double().chunk(2, dim=-1)
            return {"normed": _exact_norm(summed, s["norm"]), "residual": summed, "query": _exact_rotate(q, c, sn),
                    "cache": cache, "mlp": gate * torch.sigmoid(gate) * up}
        if case["kind"] == "edges":
            tokens = torch.stack([row.argmax() for row in s["logits"].double()])
            rows = s["embedding"][tokens].double()
            return {"tokens": None, "residual": rows, "normed": _exact_norm(rows, s["weight"])}
        return _exact_model(case, s)


def _exact_model(case, s):
    model, m, n = s["model"], s["metadata"], case["decodes"]
    inverse = 1.0 / (model.config.rope_theta ** (torch.arange(0, 128, 2, dtype=torch.float64, device=s["ids"].device) / 128))
    angles = torch.outer(m.query_positions.double(), inverse)
    angles = torch.cat((angles, angles), dim=-1)[:, None]
    c, sn = angles.cos(), angles.sin()
    x = model.embed[s["ids"]].double()
    for layer, cache in zip(model.layers, s["caches"]):
        qkv = _exact_norm(x, layer["input_norm"]) @ layer["qkv"].double().t().contiguous()
        q, k, v = qkv[:, :2048].view(n, 16, 128), qkv[:, 2048:3072].view(n, 8, 128), qkv[:, 3072:].view(n, 8, 128)
        q = _exact_rotate(_exact_norm(q, layer["q_norm"]), c, sn)
        k = _exact_rotate(_exact_norm(k, layer["k_norm"]), c, sn)
        attended = _exact_attention(case, q, k, v, cache.double(), m.block_table, m.slot_mapping, m.context_lengths,
                                    16, 8, 128)
        x = x + attended.flatten(1) @ layer["o"].double().t().contiguous()
        gate_up = _exact_norm(x, layer["post_norm"]) @ layer["gate_up"].double().t().contiguous()
        gate, up = gate_up.chunk(2, dim=-1)
        x = x + (gate * torch.sigmoid(gate) * up) @ layer["down"].double().t().contiguous()
    logits = _exact_norm(x, model.final_norm) @ model.lm_head.double().t().contiguous()
    return {"logits": logits, "caches": [None for _ in s["caches"]]}
