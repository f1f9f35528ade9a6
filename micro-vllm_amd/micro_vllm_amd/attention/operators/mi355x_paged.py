"""The gfx950 paged-attention operator (registered as ``"mi355x_paged"``).

Drop-in for the reference's attention operators
(src/micro_vllm/attention/operators/reference.py:11-81,
triton_paged.py:392-418): same positional signature, same in-place cache
write, a new output tensor like ``query``. All work runs in the HIP library
through its C ABI on the current torch stream; nothing here synchronises
with the host, so a forward can be captured in a HIP graph.

Error conventions follow the reference: tensors off the GPU raise
``RuntimeError``; an unsupported dtype raises ``ValueError``.
"""

from __future__ import annotations

import math

import torch

from micro_vllm_amd import _native
from micro_vllm_amd.attention.attention import AttentionMetadata
from micro_vllm_amd.attention.operators.base import AttentionOperator

SUPPORTED_DTYPES = (torch.bfloat16, torch.float16, torch.float32)


_INT64 = torch.int64


def _index(t: torch.Tensor, name: str, device: torch.device) -> torch.Tensor:
    if t.dtype is not _INT64:
        raise ValueError(f"metadata.{name} must be int64, got {t.dtype}")
    if t.device != device:
        raise RuntimeError(f"metadata.{name} is on {t.device}, expected {device}")
    return t if t.is_contiguous() or t.dim() != 1 else t.contiguous()


def _batch_fields(metadata: AttentionMetadata, device: torch.device) -> tuple[tuple, tuple, tuple, int, int, tuple]:
    """(pointers, (tokens, requests, table width), table strides, block size,
    max_query_len) of ``metadata`` in ``Batch`` order, checked; and the tensors
    whose memory the pointers name (made contiguous where they were not)."""

    positions = _index(metadata.query_positions, "query_positions", device)
    starts = _index(metadata.query_context_start_positions, "query_context_start_positions", device)
    qsl = _index(metadata.query_start_locations, "query_start_locations", device)
    lengths = _index(metadata.context_lengths, "context_lengths", device)
    slots = _index(metadata.slot_mapping, "slot_mapping", device)
    table = _index(metadata.block_table, "block_table", device)
    if table.dim() != 2:
        raise ValueError(f"metadata.block_table must be 2-D, got shape {tuple(table.shape)}")
    num_requests = lengths.numel()
    if qsl.numel() != num_requests + 1:
        raise ValueError(
            f"query_start_locations has {qsl.numel()} entries for {num_requests} requests"
        )
    rows, width = table.shape
    if rows < num_requests:
        raise ValueError(f"block_table has {rows} rows for {num_requests} requests")
    num_tokens = positions.numel()
    if starts.numel() != num_tokens or slots.numel() != num_tokens:
        raise ValueError("query positions, context starts and slot_mapping differ in length")
    hint = getattr(metadata, "max_query_len", None)
    return (
        (
            positions.data_ptr() if num_tokens else 0,
            starts.data_ptr() if num_tokens else 0,
            qsl.data_ptr(),
            lengths.data_ptr() if num_requests else 0,
            table.data_ptr() if rows and width else 0,
            slots.data_ptr() if num_tokens else 0,
        ),
        (num_tokens, num_requests, width),
        table.stride(),
        metadata.block_size,
        hint if hint is not None else -1,
        (positions, starts, qsl, lengths, slots, table),
    )


def batch_descriptor(metadata: AttentionMetadata, device: torch.device) -> tuple[_native.Batch, list]:
    """C-ABI view of ``metadata``; the list keeps any made-contiguous copies alive."""

    *fields, keep = _batch_fields(metadata, device)
    return _native.Batch.from_buffer_copy(_native.pack_batch(*fields)), list(keep)


def _check_inputs(
    query: torch.Tensor,
    key: torch.Tensor,
    value: torch.Tensor,
    layer_kv_cache: torch.Tensor,
    metadata: AttentionMetadata,
) -> None:
    if query.device.type != "cuda":
        raise RuntimeError("mi355x_paged attention requires GPU tensors")
    if query.dtype not in SUPPORTED_DTYPES:
        raise ValueError(
            "mi355x_paged attention supports torch.bfloat16, torch.float16 and torch.float32, "
            f"got {query.dtype}"
        )
    device, dtype = query.device, query.dtype
    for name, t in (("key", key), ("value", value), ("layer_kv_cache", layer_kv_cache)):
        if t.device != device:
            raise RuntimeError(f"{name} is on {t.device}, query on {device}")
        if t.dtype != dtype:
            raise ValueError(f"{name} dtype {t.dtype} differs from query dtype {dtype}")
    if layer_kv_cache.dim() != 5 or layer_kv_cache.shape[2] != metadata.block_size:
        raise ValueError(
            f"layer_kv_cache shape {tuple(layer_kv_cache.shape)} does not match block_size "
            f"{metadata.block_size}"
        )
    if key.shape[0] != query.shape[0] or value.shape != key.shape:
        raise ValueError("query, key and value must have the same number of tokens")
    if query.shape[1] % key.shape[1] != 0:
        raise ValueError("query heads must be a multiple of key/value heads")


def hip_write_kv_cache(
    key: torch.Tensor,
    value: torch.Tensor,
    layer_kv_cache: torch.Tensor,
    metadata: AttentionMetadata,
) -> None:
    """Scatter K/V into their cache slots (bit-exact; slot -1 writes nothing)."""

    device = layer_kv_cache.device
    if device.type != "cuda":
        raise RuntimeError("mi355x_paged cache writes require GPU tensors")
    slots = _index(metadata.slot_mapping, "slot_mapping", device)
    if slots.numel() != key.shape[0]:
        raise ValueError("slot_mapping length differs from the number of key rows")
    lib = _native.load()
    _native.check(
        lib.mvllm_kv_write(
            _native.tensor3(key),
            _native.tensor3(value),
            _native.kv_cache(layer_kv_cache),
            slots.data_ptr() if slots.numel() else None,
            key.shape[0],
            _native.stream_handle(device),
        ),
        "mvllm_kv_write",
    )


def hip_paged_attention(
    query: torch.Tensor,
    key: torch.Tensor,
    value: torch.Tensor,
    layer_kv_cache: torch.Tensor,
    metadata: AttentionMetadata,
    *,
    timing: _native.Timing | None = None,
) -> torch.Tensor:
    """Write current K/V, then ragged causal attention through the block table.

    ``timing`` (measurement only) carries hipEvent_t handles recorded around
    the decode and prefill kernel launches.
    """

    _check_inputs(query, key, value, layer_kv_cache, metadata)
    device = query.device
    *fields, keep = _batch_fields(metadata, device)
    batch = _native.pack_batch(*fields)
    output = torch.empty_like(query)
    _, num_heads, head_dim = query.shape
    workspace_bytes = _native.packed("mvllm_attention_workspace_bytes")(batch, num_heads, head_dim)
    workspace = torch.empty(max(workspace_bytes, 1), dtype=torch.uint8, device=device)
    scale = 1.0 / math.sqrt(head_dim)
    stream = _native.stream_handle(device)
    if timing is None:
        status = _native.packed("mvllm_attention_forward")(
            _native.pack_tensor3(query),
            _native.pack_tensor3(key),
            _native.pack_tensor3(value),
            _native.pack_kv_cache(layer_kv_cache),
            batch,
            _native.pack_tensor3(output),
            scale,
            workspace.data_ptr(),
            max(workspace_bytes, 1),
            stream,
        )
    else:
        status = _native.load().mvllm_attention_forward_timed(
            _native.tensor3(query),
            _native.tensor3(key),
            _native.tensor3(value),
            _native.kv_cache(layer_kv_cache),
            _native.Batch.from_buffer_copy(batch),
            _native.tensor3(output),
            scale,
            workspace.data_ptr(),
            workspace.numel(),
            timing,
            stream,
        )
    _native.check(status, "mvllm_attention_forward")
    del keep
    return output


def plan_geometry(layer_kv_cache: torch.Tensor) -> tuple:
    """What a plan takes from the cache: the element type, block size, KV heads,
    head_dim, strides within a block and alignment decide which kernels run and
    how the decode splits, their counters and the query blocks are laid out.
    The block count and the memory itself do not matter."""

    return (
        layer_kv_cache.dtype,
        *layer_kv_cache.shape[2:],
        *layer_kv_cache.stride()[1:],
        layer_kv_cache.stride(0) * layer_kv_cache.element_size() % 16,
        layer_kv_cache.data_ptr() % 16,
    )


class AttentionPlan:
    """Work lists of one batch, built once and shared by every layer of a step.

    The reference's operator runs per layer (qwen.py:89-99); the lists depend
    only on the batch, the query heads and the cache's geometry, so a model
    whose layers share one metadata bundle and one geometry plans once per step
    (``mvllm_attention_plan``) and each layer's
    ``hip_attention_over_cache(..., plan=plan)`` skips the list kernels. A
    layer whose cache differs (``plan_geometry``) is answered through lists of
    its own. The plan owns the workspace, which every planned call reuses for
    its split-KV partials and the counters of its finished splits: planned
    calls of one plan run in one stream and never overlap.
    """

    def __init__(self, metadata: AttentionMetadata, num_q_heads: int, layer_kv_cache: torch.Tensor):
        device = layer_kv_cache.device
        if device.type != "cuda":
            raise RuntimeError("mi355x_paged attention plans require a GPU cache")
        self.metadata = metadata
        self.num_q_heads = num_q_heads
        self.geometry = plan_geometry(layer_kv_cache)
        self.batch, self._keep = batch_descriptor(metadata, device)
        lib = _native.load()
        head_dim = layer_kv_cache.shape[-1]
        nbytes = lib.mvllm_attention_workspace_bytes(self.batch, num_q_heads, head_dim)
        self.workspace = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=device)
        _native.check(
            lib.mvllm_attention_plan(
                self.batch,
                num_q_heads,
                _native.kv_cache(layer_kv_cache),
                self.workspace.data_ptr(),
                self.workspace.numel(),
                _native.stream_handle(device),
            ),
            "mvllm_attention_plan",
        )


def hip_attention_over_cache(
    query: torch.Tensor,
    layer_kv_cache: torch.Tensor,
    metadata: AttentionMetadata,
    plan: AttentionPlan | None = None,
) -> torch.Tensor:
    """Ragged causal attention over a cache that already holds the step's
    K/V (written by ``layers.qk_norm_rope_kv_write``): the attention part of
    ``hip_paged_attention``, without the cache write. With ``plan`` (made for
    this metadata and head count) the work lists are not rebuilt, unless the
    cache's geometry is not the one that the plan was made for."""

    if query.device.type != "cuda" or layer_kv_cache.device != query.device:
        raise RuntimeError("mi355x_paged attention requires GPU tensors on one device")
    if query.dtype not in SUPPORTED_DTYPES or layer_kv_cache.dtype != query.dtype:
        raise ValueError(f"unsupported or mismatched dtypes {query.dtype} / {layer_kv_cache.dtype}")
    device = query.device
    output = torch.empty_like(query)
    lib = _native.load()
    if plan is not None:
        if plan.metadata is not metadata or plan.num_q_heads != query.shape[1]:
            raise ValueError("attention plan was made for other metadata or another head count")
        if plan.geometry != plan_geometry(layer_kv_cache):
            plan = None
    if plan is not None:
        batch, keep, workspace, entry = plan.batch, None, plan.workspace, "mvllm_paged_attention_planned"
    else:
        batch, keep = batch_descriptor(metadata, device)
        workspace_bytes = lib.mvllm_attention_workspace_bytes(batch, query.shape[1], query.shape[2])
        workspace = torch.empty(max(workspace_bytes, 1), dtype=torch.uint8, device=device)
        entry = "mvllm_paged_attention"
    _native.check(
        getattr(lib, entry)(
            _native.tensor3(query),
            _native.kv_cache(layer_kv_cache),
            batch,
            _native.tensor3(output),
            1.0 / math.sqrt(query.shape[-1]),
            workspace.data_ptr(),
            workspace.numel(),
            _native.stream_handle(device),
        ),
        entry,
    )
    del keep
    return output


def hip_gather_kv_cache(
    layer_kv_cache: torch.Tensor,
    metadata: AttentionMetadata,
    capacity: int | None = None,
) -> tuple[torch.Tensor, torch.Tensor]:
    """Padded ``[requests, capacity, heads, dim]`` K and V histories (bit-exact).

    Row ``i`` of request ``r`` holds position ``start(first query) + i``;
    rows past the request's context are left as allocated (zeros here).
    ``capacity`` defaults to ``block_table.shape[1] * block_size``.
    """

    device = layer_kv_cache.device
    if device.type != "cuda":
        raise RuntimeError("mi355x_paged gathers require GPU tensors")
    batch, keep = batch_descriptor(metadata, device)
    if capacity is None:
        capacity = metadata.block_table.shape[1] * metadata.block_size
    shape = (metadata.num_requests, capacity, *layer_kv_cache.shape[3:])
    keys = torch.zeros(shape, dtype=layer_kv_cache.dtype, device=device)
    values = torch.zeros(shape, dtype=layer_kv_cache.dtype, device=device)
    lib = _native.load()
    _native.check(
        lib.mvllm_gather_kv(
            _native.kv_cache(layer_kv_cache),
            batch,
            capacity,
            keys.data_ptr() if keys.numel() else None,
            values.data_ptr() if values.numel() else None,
            _native.stream_handle(device),
        ),
        "mvllm_gather_kv",
    )
    del keep
    return keys, values


class MI355XPagedAttentionOperator(AttentionOperator):
    """gfx950 HIP paged attention: split-KV MFMA decode + MFMA prefill."""

    def forward(
        self,
        query: torch.Tensor,
        key: torch.Tensor,
        value: torch.Tensor,
        layer_kv_cache: torch.Tensor,
        metadata: AttentionMetadata,
        /,
    ) -> torch.Tensor:
        return hip_paged_attention(
            query,
            key,
            value,
            layer_kv_cache,
            metadata,
        )
