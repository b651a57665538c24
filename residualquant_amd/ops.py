"""Operator surface of the packed KV-cache path on MI355X.

``quantize`` and ``attention`` keep the reference ops' signatures, keyword
names, in-place semantics and error messages
(plugins/residual_quantization/csrc/dispatch/binding.cpp:19-38;
validation quantize/api.cpp:18-85, attention/api.cpp:23-104,
common/api.h:42-64, dispatch/kernel_registry.h:42-72).  Tensor checks that a
pointer interface cannot see (device, dtype, strides) run here and raise
``RuntimeError``; everything else is checked by ``librq_hip.so`` before any
device work.  Work is enqueued on the current HIP stream of the cache's
device; nothing synchronizes.
"""

from __future__ import annotations

import ctypes
from contextlib import nullcontext
from functools import lru_cache
from typing import Optional, Sequence, Tuple

import torch

from . import _lib

_MODES = {"anchor": 0, "adjacent": 1}
_COEFFICIENTS = {"unit": 0, "norm": 1, "ls": 2}


def _require(condition: bool, message: str) -> None:
    if not condition:
        raise RuntimeError(message)


# A call on one small request runs about 14 us on the GPU, and what the host
# does per call is what a loop of such calls waits for (20 us per attention
# call before the checks below read each tensor's shape and strides once, the
# device context was entered only for another device than the current one, the
# schedule's C arrays were kept by value and the stream's handle was read
# without a Stream object; 14 us, the GPU time, with them).


def _validate_bf16_token_tensor(tensor: torch.Tensor) -> Tuple[torch.Size, int]:
    """The tensor's shape and token stride."""
    # common/api.h:42-49
    if tensor.is_cuda and tensor.dtype is torch.bfloat16:
        shape = tensor.shape
        if len(shape) == 3:
            stride = tensor.stride()
            if stride[1] == shape[2] and stride[2] == 1:
                return shape, stride[0]
    raise RuntimeError("BF16 [tokens, heads, channels] with packed trailing strides required")


def _rotation_pointer(rotation: Optional[torch.Tensor], device: int, heads: int, head_dim: int):
    # common/api.h:51-64
    if rotation is None:
        return None
    _require(rotation.get_device() == device and rotation.is_contiguous() and rotation.dtype is torch.float16
             and rotation.shape == (heads, head_dim, head_dim),
             "Contiguous FP16 [heads, channels, channels] rotation required")
    return rotation.data_ptr()


@lru_cache(maxsize=64)
def _schedule_arrays(records: Tuple[Tuple[int, int], ...]):
    # The library only reads them.
    bits = (ctypes.c_int * max(1, len(records)))(*[r[0] for r in records])
    groups = (ctypes.c_int * max(1, len(records)))(*[r[1] for r in records])
    return bits, groups, ctypes.addressof(bits), ctypes.addressof(groups)


def _schedule(records: Sequence[Sequence[int]]):
    """(bits, groups, their addresses) of a schedule; the arrays live as long as the caller holds them."""
    return _schedule_arrays(tuple([(int(r[0]), int(r[1])) for r in records]))


def _on_device(device: int):
    """A context on CUDA device ``device`` (nothing to do where it is current)."""
    return nullcontext() if torch.cuda.current_device() == device else torch.cuda.device(device)


def _stream(device: int) -> int:
    return torch._C._cuda_getCurrentRawStream(device)


def quantize(key_value_pairs: Sequence[Tuple[torch.Tensor, torch.Tensor]], kv_cache: torch.Tensor,
             slot_mapping: torch.Tensor, key_rotation: Optional[torch.Tensor],
             value_rotation: Optional[torch.Tensor], key_mean: Optional[torch.Tensor],
             records: Sequence[Sequence[int]], reference_mode: str, anchor_index: int,
             coefficient_method: str) -> None:
    """Quantize one completed loop group into the packed paged cache, in place.

    Mirrors quantize() (quantize/api.cpp:8-95): ``key_value_pairs[r]`` holds
    the BF16 [tokens, heads, D] K/V of record r in loop order; token i goes to
    cache slot ``slot_mapping[i]`` (negative = skipped).
    """
    _require(len(records) > 0 and len(key_value_pairs) == len(records),
             "A nonempty group with one K/V input per record required")
    _require(kv_cache.is_cuda and kv_cache.dtype == torch.uint8 and kv_cache.is_contiguous()
             and kv_cache.dim() == 5 and kv_cache.size(0) == 2,
             "Contiguous CUDA UINT8 [2, blocks, heads, page tokens, page width] cache required")
    device = kv_cache.get_device()
    _, num_blocks, heads, page_tokens, page_width = kv_cache.shape
    head_dim = key_value_pairs[0][0].size(-1)
    _require(slot_mapping.get_device() == device and slot_mapping.dtype is torch.int64
             and slot_mapping.dim() == 1 and slot_mapping.is_contiguous(),
             "Contiguous INT64 slot mapping on the cache device required")
    tokens = slot_mapping.numel()
    pointers, strides, input_rows = ([], []), ([], []), None
    for pair in key_value_pairs:
        layouts = []
        for tensor in pair:
            shape, stride = _validate_bf16_token_tensor(tensor)
            rows = shape[0]
            _require(tensor.get_device() == device and shape[1] == heads and shape[2] == head_dim,
                     "K/V must match the cache device/head count and logical channel count")
            _require(rows >= tokens, "Input has fewer rows than slot mapping")
            layouts.append((tensor.data_ptr(), stride, rows))
        for plane in (0, 1):
            pointer, stride, rows = layouts[plane]
            pointers[plane].append(pointer)
            strides[plane].append(stride)
            input_rows = rows if input_rows is None or rows < input_rows else input_rows
    if key_mean is not None:
        _require(key_mean.get_device() == device and key_mean.dtype is torch.float32
                 and key_mean.is_contiguous() and key_mean.dim() == 3
                 and key_mean.size(0) == len(records) and key_mean.size(1) == heads
                 and key_mean.size(2) == head_dim,
                 "Contiguous FP32 [records, heads, channels] key mean required")
    key_rotation_ptr = _rotation_pointer(key_rotation, device, heads, head_dim)
    value_rotation_ptr = _rotation_pointer(value_rotation, device, heads, head_dim)
    _require(coefficient_method in _COEFFICIENTS, "Unsupported coefficient")
    _require(reference_mode in _MODES, f"Unknown packed reference mode: {reference_mode}")

    count = len(records)
    pointer_array, stride_array = ctypes.c_void_p * count, ctypes.c_int64 * count
    keys, values = pointer_array(*pointers[0]), pointer_array(*pointers[1])
    key_strides, value_strides = stride_array(*strides[0]), stride_array(*strides[1])
    schedule = _schedule(records)
    with _on_device(device):
        status = _lib.lib().rq_quantize(
            count, ctypes.addressof(keys), ctypes.addressof(key_strides), ctypes.addressof(values),
            ctypes.addressof(value_strides), input_rows, kv_cache.data_ptr(), num_blocks, heads, page_tokens,
            page_width, slot_mapping.data_ptr(), tokens, head_dim, key_rotation_ptr, value_rotation_ptr,
            key_mean.data_ptr() if key_mean is not None else None, schedule[2], schedule[3],
            _MODES[reference_mode], int(anchor_index), _COEFFICIENTS[coefficient_method], _stream(device))
    _lib.check(status)


def attention_workspace_bytes(rows: int, heads: int, head_dim: int, max_pages: int,
                              page_tokens: int) -> int:
    """Device workspace (bytes) for ``attention``; depends on shapes only.  (A
    smaller one that holds what the call's route requires is taken as well.)"""
    return int(_lib.lib().rq_attention_workspace_bytes(rows, heads, head_dim, max_pages, page_tokens))


def _workspace(workspace: Optional[torch.Tensor], needed: int, device) -> torch.Tensor:
    if workspace is None:
        return torch.empty(needed, dtype=torch.uint8, device=device)
    # (The library refuses one that is too small for the call's route.)
    _require(workspace.is_cuda and workspace.device == device and workspace.is_contiguous(),
             f"Attention workspace of {needed} bytes required")
    return workspace


def _validate_attention_inputs(query, key, value, output, query_start_loc, seq_lens, block_table):
    """The token strides of query, key, value and output."""
    shape, query_stride = _validate_bf16_token_tensor(query)
    device = query.get_device()
    strides = [query_stride]
    for tensor in (key, value, output):
        other, stride = _validate_bf16_token_tensor(tensor)
        _require(tensor.get_device() == device and other == shape,
                 "Q/K/V/output must have matching shapes and devices")
        strides.append(stride)
    _require(query.data_ptr() % 8 == 0 and query_stride % 4 == 0 and key.data_ptr() % 8 == 0 and strides[1] % 4 == 0,
             "Q/K addresses and token strides must be 8-byte aligned")
    requests = seq_lens.numel()
    _require(query_start_loc.get_device() == device and query_start_loc.dtype is torch.int32
             and query_start_loc.dim() == 1 and query_start_loc.is_contiguous()
             and query_start_loc.numel() == requests + 1,
             "Contiguous INT32 query starts with one final boundary required")
    _require(seq_lens.get_device() == device and seq_lens.dtype is torch.int32
             and seq_lens.dim() == 1 and seq_lens.is_contiguous(),
             "Contiguous INT32 sequence lengths required")
    _require(block_table.get_device() == device and block_table.dtype is torch.int32
             and block_table.dim() == 2 and block_table.stride(1) == 1
             and block_table.size(0) >= requests,
             "INT32 page table with packed rows required")
    return strides


def attention(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor, kv_cache: torch.Tensor,
              output: torch.Tensor, query_start_loc: torch.Tensor, seq_lens: torch.Tensor,
              block_table: torch.Tensor, key_rotation: Optional[torch.Tensor],
              value_rotation: Optional[torch.Tensor], key_mean: Optional[torch.Tensor],
              records: Sequence[Sequence[int]], reference_mode: str, anchor_index: int,
              loop_index: int, workspace: Optional[torch.Tensor] = None) -> None:
    """Paged decode attention of loop ``loop_index`` over the packed cache, writing ``output``.

    Mirrors attention() (attention/api.cpp:8-115).  ``key``/``value`` are the
    current token's K/V (not yet in the cache).  ``workspace`` (optional, not
    in the reference) lets a caller reuse one device buffer of
    ``attention_workspace_bytes(...)`` bytes, e.g. across graph replays.
    """
    strides, key_rotation_ptr, value_rotation_ptr = _validate_packed_inputs(
        query, key, value, kv_cache, output, query_start_loc, seq_lens, block_table, key_rotation, value_rotation,
        key_mean, records, reference_mode, loop_index)
    _call_packed_attention(_lib.lib().rq_attention, strides, query, key, value, kv_cache, output, query_start_loc,
                           seq_lens, block_table, key_rotation_ptr, value_rotation_ptr, key_mean, records,
                           reference_mode, anchor_index, loop_index, workspace)


def _validate_packed_inputs(query, key, value, kv_cache, output, query_start_loc, seq_lens, block_table,
                            key_rotation, value_rotation, key_mean, records, reference_mode, loop_index):
    strides = _validate_attention_inputs(query, key, value, output, query_start_loc, seq_lens, block_table)
    _, heads, head_dim = query.shape
    device = query.get_device()
    _require(kv_cache.get_device() == device and kv_cache.dtype is torch.uint8
             and kv_cache.is_contiguous() and kv_cache.dim() == 5 and kv_cache.size(0) == 2
             and kv_cache.size(2) == heads,
             "Contiguous UINT8 KV cache on the query device required")
    if key_mean is not None:
        _require(key_mean.get_device() == device and key_mean.dtype is torch.float32
                 and key_mean.is_contiguous() and key_mean.data_ptr() % 16 == 0
                 and key_mean.numel() == len(records) * heads * head_dim,
                 "16-byte aligned contiguous FP32 key mean with matching dimensions required")
    value_rotation_ptr = _rotation_pointer(value_rotation, device, heads, head_dim)
    key_rotation_ptr = _rotation_pointer(key_rotation, device, heads, head_dim)
    _require(key_rotation_ptr is None or key_rotation_ptr % 16 == 0,
             "16-byte aligned key rotation required for asynchronous copies")
    _require(0 <= loop_index < len(records), "Invalid loop index")
    _require(reference_mode in _MODES, f"Unknown packed reference mode: {reference_mode}")
    return strides, key_rotation_ptr, value_rotation_ptr


def packed_prefill_attention(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor,
                             kv_cache: torch.Tensor, output: torch.Tensor, query_start_loc: torch.Tensor,
                             seq_lens: torch.Tensor, block_table: torch.Tensor,
                             key_rotation: Optional[torch.Tensor], value_rotation: Optional[torch.Tensor],
                             key_mean: Optional[torch.Tensor], records: Sequence[Sequence[int]],
                             reference_mode: str, anchor_index: int, loop_index: int,
                             workspace: Optional[torch.Tensor] = None) -> None:
    """Attention of each request's last n tokens (its query rows) over its packed history.

    Request b's rows ``query_start_loc[b]..query_start_loc[b+1]`` are the
    last n of its ``seq_lens[b]`` tokens: they attend to the first
    ``seq_lens[b] - n`` tokens from the cache and, causally, to the request's
    own new ``key``/``value`` rows (row r sees new rows 0..r).  This is the
    prefill of a prompt chunk over a packed prefix, which the reference
    cannot run (its scheduler forbids partial prefill, rq/scheduler.py:11-18);
    arguments and validation are those of ``attention`` (head_dim 96 or
    128, anchor or adjacent mode); a request may have no new rows.
    """
    strides, key_rotation_ptr, value_rotation_ptr = _validate_packed_inputs(
        query, key, value, kv_cache, output, query_start_loc, seq_lens, block_table, key_rotation, value_rotation,
        key_mean, records, reference_mode, loop_index)
    _call_packed_attention(_lib.lib().rq_packed_prefill_attention, strides, query, key, value, kv_cache, output,
                           query_start_loc, seq_lens, block_table, key_rotation_ptr, value_rotation_ptr, key_mean,
                           records, reference_mode, anchor_index, loop_index, workspace)


def _call_packed_attention(function, strides, query, key, value, kv_cache, output, query_start_loc, seq_lens,
                           block_table, key_rotation_ptr, value_rotation_ptr, key_mean, records, reference_mode,
                           anchor_index, loop_index, workspace):
    rows, heads, head_dim = query.shape
    _, num_blocks, _, page_tokens, page_width = kv_cache.shape
    max_pages = block_table.size(1)
    device = query.get_device()
    ws = _workspace(workspace, attention_workspace_bytes(rows, heads, head_dim, max_pages, page_tokens), query.device)
    schedule = _schedule(records)
    with _on_device(device):
        status = function(
            query.data_ptr(), strides[0], key.data_ptr(), strides[1], value.data_ptr(), strides[2],
            output.data_ptr(), strides[3], rows, heads, head_dim, kv_cache.data_ptr(), num_blocks, page_tokens,
            page_width, query_start_loc.data_ptr(), seq_lens.data_ptr(), seq_lens.numel(), block_table.data_ptr(),
            block_table.stride(0), max_pages, key_rotation_ptr, value_rotation_ptr,
            key_mean.data_ptr() if key_mean is not None else None, len(records), schedule[2], schedule[3],
            _MODES[reference_mode], int(anchor_index), int(loop_index), ws.data_ptr(),
            ws.numel() * ws.element_size(), _stream(device))
    _lib.check(status)


def dequantize(kv_cache: torch.Tensor, slots: torch.Tensor, head_dim: int,
               key_mean: Optional[torch.Tensor], records: Sequence[Sequence[int]],
               reference_mode: str, anchor_index: int, loop_index: int):
    """Restored BF16 K and V [tokens, heads, D] of ``loop_index`` at ``slots`` (rotated space).

    The record value both reference kernels reconstruct internally
    (quantize/kernel.cuh:160-203, attention/compute.cuh:28-197).
    """
    _require(kv_cache.is_cuda and kv_cache.dtype == torch.uint8 and kv_cache.is_contiguous()
             and kv_cache.dim() == 5 and kv_cache.size(0) == 2,
             "Contiguous CUDA UINT8 [2, blocks, heads, page tokens, page width] cache required")
    _require(slots.device == kv_cache.device and slots.dtype == torch.int64 and slots.dim() == 1
             and slots.is_contiguous(), "Contiguous INT64 slot mapping on the cache device required")
    heads = kv_cache.size(2)
    if key_mean is not None:
        _require(key_mean.device == kv_cache.device and key_mean.dtype == torch.float32
                 and key_mean.is_contiguous() and key_mean.numel() == len(records) * heads * head_dim,
                 "Contiguous FP32 [records, heads, channels] key mean required")
    _require(reference_mode in _MODES, f"Unknown packed reference mode: {reference_mode}")
    key_out = torch.empty((slots.numel(), heads, head_dim), dtype=torch.bfloat16, device=kv_cache.device)
    value_out = torch.empty_like(key_out)
    schedule = _schedule(records)
    device = kv_cache.get_device()
    with _on_device(device):
        status = _lib.lib().rq_dequantize(
            kv_cache.data_ptr(), kv_cache.size(1), heads, kv_cache.size(3), kv_cache.size(4),
            slots.data_ptr(), slots.numel(), head_dim,
            key_mean.data_ptr() if key_mean is not None else None, len(records),
            schedule[2], schedule[3],
            _MODES[reference_mode], int(anchor_index), int(loop_index), key_out.data_ptr(),
            value_out.data_ptr(), _stream(device))
    _lib.check(status)
    return key_out, value_out


def paged_attention_bf16(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor,
                         cache: torch.Tensor, output: torch.Tensor, query_start_loc: torch.Tensor,
                         seq_lens: torch.Tensor, block_table: torch.Tensor,
                         workspace: Optional[torch.Tensor] = None) -> None:
    """BF16 paged decode attention over ``cache`` [2, blocks, heads, PT, D] (the baseline)."""
    _validate_attention_inputs(query, key, value, output, query_start_loc, seq_lens, block_table)
    heads, head_dim = query.size(1), query.size(2)
    _require(cache.device == query.device and cache.dtype == torch.bfloat16 and cache.is_contiguous()
             and cache.dim() == 5 and cache.size(0) == 2 and cache.size(2) == heads
             and cache.size(4) == head_dim,
             "Contiguous BF16 [2, blocks, heads, page tokens, channels] cache required")
    rows = query.size(0)
    max_pages = block_table.size(1)
    needed = attention_workspace_bytes(rows, heads, head_dim, max_pages, cache.size(3))
    ws = _workspace(workspace, needed, query.device)
    device = query.get_device()
    with _on_device(device):
        status = _lib.lib().rq_paged_attention_bf16(
            query.data_ptr(), query.stride(0), key.data_ptr(), key.stride(0), value.data_ptr(),
            value.stride(0), output.data_ptr(), output.stride(0), rows, heads, head_dim,
            cache.data_ptr(), cache.size(1), cache.size(3), query_start_loc.data_ptr(),
            seq_lens.data_ptr(), seq_lens.numel(), block_table.data_ptr(), block_table.stride(0),
            max_pages, ws.data_ptr(), ws.numel() * ws.element_size(), _stream(device))
    _lib.check(status)


def flash_attn_varlen_func(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, max_seqlen_q: int,
                           cu_seqlens_q: torch.Tensor, max_seqlen_k: int,
                           cu_seqlens_k: Optional[torch.Tensor] = None, dropout_p: float = 0.0,
                           softmax_scale: Optional[float] = None, causal: bool = False,
                           window_size=None, softcap: float = 0.0, alibi_slopes=None,
                           deterministic: bool = False, return_attn_probs: bool = False,
                           block_table=None, return_softmax_lse: bool = False,
                           out: Optional[torch.Tensor] = None, fa_version=None) -> torch.Tensor:
    """Varlen (causal) attention over raw BF16 Q/K/V, the full-prompt branch.

    Drop-in for the ``flash_attn_varlen_func`` call of the reference backend
    (src/residual_quantization/packed_backend.py:63-77, vLLM 0.10.2): q
    [tokens_q, heads_q, D], k/v [tokens_k, heads_k, D] BF16, sequence s spans
    cu_seqlens[s]..cu_seqlens[s+1]; with ``causal`` query i of a sequence sees
    keys j <= i + len_k - len_q.  The features that call does not use
    (dropout, windows, softcap, ALiBi, paged K/V, returned LSE or
    probabilities) raise.  ``fa_version`` is accepted and ignored.
    """
    _require(dropout_p == 0.0 and softcap == 0.0 and alibi_slopes is None and block_table is None
             and not return_attn_probs and not return_softmax_lse
             and (window_size is None or tuple(window_size) == (-1, -1)),
             "Only dropout-free, unwindowed attention without ALiBi, softcap, paged K/V or returned "
             "LSE is supported")
    cu_seqlens_k = cu_seqlens_q if cu_seqlens_k is None else cu_seqlens_k
    (q_shape, q_stride), (k_shape, k_stride), (v_shape, v_stride) = map(_validate_bf16_token_tensor, (q, k, v))
    device = q.get_device()
    _require(k.get_device() == device and v.get_device() == device and k_shape == v_shape
             and k_shape[2] == q_shape[2], "Q/K/V must share device and head_dim; K and V must match")
    if out is None:
        out = torch.empty_like(q)
    out_shape, out_stride = _validate_bf16_token_tensor(out)
    _require(out.get_device() == device and out_shape == q_shape, "out must match q")
    for seqlens in (cu_seqlens_q, cu_seqlens_k):
        _require(seqlens.get_device() == device and seqlens.dtype is torch.int32 and seqlens.dim() == 1
                 and seqlens.is_contiguous(), "Contiguous INT32 cu_seqlens on the Q device required")
    _require(cu_seqlens_q.numel() == cu_seqlens_k.numel() and cu_seqlens_q.numel() >= 1,
             "cu_seqlens_q and cu_seqlens_k must describe the same sequences")
    _, heads_q, head_dim = q_shape
    scale = head_dim ** -0.5 if softmax_scale is None else float(softmax_scale)
    batch = cu_seqlens_q.numel() - 1
    same = cu_seqlens_q.data_ptr() == cu_seqlens_k.data_ptr()
    needed = _lib.lib().rq_prefill_workspace_bytes(batch, heads_q, head_dim, int(max_seqlen_q),
                                                   int(max_seqlen_k), 1 if causal else 0, 1 if same else 0)
    workspace = torch.empty(max(needed, 1), dtype=torch.uint8, device=q.device)
    with _on_device(device):
        status = _lib.lib().rq_prefill_attention(
            q.data_ptr(), q_stride, k.data_ptr(), k_stride, v.data_ptr(), v_stride, out.data_ptr(), out_stride,
            heads_q, k_shape[1], head_dim, cu_seqlens_q.data_ptr(), cu_seqlens_k.data_ptr(), batch,
            int(max_seqlen_q), int(max_seqlen_k), scale, 1 if causal else 0, workspace.data_ptr(),
            workspace.numel(), _stream(device))
    _lib.check(status)
    return out


prefill_attention = flash_attn_varlen_func


def timing_enable(enabled: bool) -> None:
    """Record HIP events around every split-K decode launch (for measurement)."""
    _lib.lib().rq_timing_enable(1 if enabled else 0)


def timing_read():
    """(milliseconds, launches) summed over the recorded split-K launches, then cleared."""
    ms = ctypes.c_double()
    launches = ctypes.c_int64()
    _lib.check(_lib.lib().rq_timing_read(ctypes.byref(ms), ctypes.byref(launches)))
    return ms.value, launches.value


def set_split_target(workgroups: int) -> None:
    """Target number of split-K workgroups per decode launch (0 restores the default)."""
    _lib.lib().rq_set_split_target(int(workgroups))
