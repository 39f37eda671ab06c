"""``paged_attention`` / ``paged_attention_prefill`` / ``paged_caching`` on torch CUDA tensors, executed by ``libinfiniop.so``.

Argument order and meaning are those of the reference's Python operators
(``python/infinicore/ops/paged_attention.py:5-40``, ``python/infinicore/ops/paged_attention_prefill.py:5-45``,
``python/infinicore/ops/paged_caching.py:5-21``).
What the reference's C++ adaptor does between that call and the C API
(``src/infinicore/ops/paged_attention/paged_attention_infiniop.cc:16-58``: build tensor descriptors,
fetch or create a cached operator descriptor keyed by the tensors' metadata, allocate a byte
workspace of the size the descriptor asks for, call the operator on the current stream) is done by ``csrc/torch_ops``
with torch providing device memory and the stream; here are the descriptors it asks for when a call's metadata is new.
"""
from __future__ import annotations

import ctypes
import importlib.util
from ctypes import c_size_t, c_void_p
from pathlib import Path

import torch

from . import libinfiniop as lib
from .libinfiniop import LIBINFINIOP, InfiniDevice, InfiniDtype, check_error

_TORCH_TO_INFINI = {
    torch.float16: InfiniDtype.F16,
    torch.bfloat16: InfiniDtype.BF16,
    torch.float32: InfiniDtype.F32,
    torch.int64: InfiniDtype.I64,
    torch.int32: InfiniDtype.I32,
    torch.uint32: InfiniDtype.U32,
    torch.uint8: InfiniDtype.U8,
    torch.int8: InfiniDtype.I8,
    torch.int16: InfiniDtype.I16,
    torch.uint16: InfiniDtype.U16,
    torch.uint64: InfiniDtype.U64,
}

_PLAN_CACHE_CAPACITY = 100  # the reference keeps a thread-local LRU of 100 descriptors per operator
_handles: dict[int, object] = {}


def _load_native():
    """csrc/torch_ops: built beside the C libraries in use, or else the one in the package's own library folder (a build of
    the C libraries alone; the extension gets their functions below, so any will do)."""
    folders = (lib.LIB_DIR, Path(__file__).resolve().parent / "lib")
    path = next((f / "_torch_ops.so" for f in folders if (f / "_torch_ops.so").is_file()), None)
    if path is None:
        raise ImportError(f"_torch_ops.so not found in {folders[0]}: build it first (python -m infinicore_amd.build, "
                          "__graft_entry__.build(), or make -C infinicore_amd/csrc torch)")
    spec = importlib.util.spec_from_file_location("infinicore_amd._torch_ops", path)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


_native = _load_native()
# the operators by number, as csrc/torch_ops/torch_ops.cc lists them
(_PAGED_ATTENTION, _PAGED_ATTENTION_PREFILL, _PAGED_CACHING, _ROPE_PAGED_CACHING, _ROPE_QK_PAGED_CACHING, _KV_CACHING) = range(6)
_RUN = ("infiniopPagedAttention", "infiniopPagedAttentionPrefill", "infiniopPagedCaching", "infiniopRoPEPagedCaching",
        "infiniopRoPEQKPagedCaching", "infiniopKVCaching")
_native.setup(tuple(ctypes.cast(getattr(LIBINFINIOP, name), c_void_p).value for name in _RUN),
              ctypes.cast(lib.LIBINFINIRT.infinirtSetDevice, c_void_p).value, int(InfiniDevice.AMD), _PLAN_CACHE_CAPACITY)


def _handle_for(index: int):
    lib.set_device(InfiniDevice.AMD, index)
    if index not in _handles:
        _handles[index] = lib.create_handle()
    return _handles[index]


def _describe(t: torch.Tensor):
    return lib.create_tensor_descriptor(tuple(t.shape), tuple(t.stride()), _TORCH_TO_INFINI[t.dtype])


class _Plan:
    """An operator descriptor, until the native cache closes it, and the bytes of scratch its calls need."""

    def __init__(self, descriptor, destroy, workspace_bytes: int):
        self.descriptor = descriptor
        self._destroy = destroy
        self.workspace_bytes = workspace_bytes
        self.descriptor_address = ctypes.cast(descriptor, c_void_p).value

    def close(self):
        if self.descriptor is not None:
            check_error(self._destroy(self.descriptor))
            self.descriptor = None


def clear_plan_cache() -> None:
    _native.clear()


def _plan(create, workspace_size, destroy, device, tensors, *more, optional=None):
    """Make the descriptor of a call: ``create(handle, &op, descriptors of the tensors.., *more)``. ``optional`` is a
    one-element tuple with a tensor that may be absent and follows the others."""
    handle = _handle_for(device.index)
    op = lib.infiniopOperatorDescriptor_t()
    descs = [_describe(t) for t in tensors]
    try:
        rest = []
        if optional is not None:
            if optional[0] is not None:
                descs.append(_describe(optional[0]))
            else:
                rest.append(lib.infiniopTensorDescriptor_t())
        check_error(getattr(LIBINFINIOP, create)(handle, ctypes.byref(op), *descs, *rest, *more), create)
    finally:
        for d in descs:
            lib.destroy_tensor_descriptor(d)
    size = c_size_t(0)
    check_error(getattr(LIBINFINIOP, workspace_size)(op, ctypes.byref(size)))
    return _Plan(op, getattr(LIBINFINIOP, destroy), size.value)


def _make_paged_attention(scale, *tensors):
    return _plan("infiniopCreatePagedAttentionDescriptor", "infiniopGetPagedAttentionWorkspaceSize",
                 "infiniopDestroyPagedAttentionDescriptor", tensors[1].device, tensors[:-1], scale, optional=tensors[-1:])


def _make_paged_attention_prefill(scale, *tensors):
    return _plan("infiniopCreatePagedAttentionPrefillDescriptor", "infiniopGetPagedAttentionPrefillWorkspaceSize",
                 "infiniopDestroyPagedAttentionPrefillDescriptor", tensors[1].device, tensors[:-1], scale,
                 optional=tensors[-1:])


def _make_paged_caching(_, *tensors):
    return _plan("infiniopCreatePagedCachingDescriptor", "infiniopGetPagedCachingWorkspaceSize",
                 "infiniopDestroyPagedCachingDescriptor", tensors[2].device, tensors)


def _make_rope_paged_caching(algo, *tensors):
    return _plan("infiniopCreateRoPEPagedCachingDescriptor", "infiniopGetRoPEPagedCachingWorkspaceSize",
                 "infiniopDestroyRoPEPagedCachingDescriptor", tensors[2].device, tensors, algo)


def _make_rope_qk_paged_caching(algo, *tensors):
    return _plan("infiniopCreateRoPEQKPagedCachingDescriptor", "infiniopGetRoPEPagedCachingWorkspaceSize",
                 "infiniopDestroyRoPEPagedCachingDescriptor", tensors[4].device, tensors, algo)


def _make_kv_caching(_, *tensors):
    return _plan("infiniopCreateKVCachingDescriptor", "infiniopGetKVCachingWorkspaceSize",
                 "infiniopDestroyKVCachingDescriptor", tensors[2].device, tensors)


def _call(operator, number, make, *tensors):
    result = _native.call(operator, number, make, *tensors)
    if type(result) is int:  # a status; otherwise the first tensor
        check_error(result, _RUN[operator])
    return result


def paged_attention(q, k_cache, v_cache, block_tables, cache_lens, alibi_slopes=None, scale: float = 1.0, *, out=None):
    """Decode attention of one query token per sequence over a paged KV pool; returns ``out``.

    q [num_seqs, num_heads, head_size]; k_cache / v_cache [num_blocks, num_kv_heads, block_size, d];
    block_tables [num_seqs, max_blocks] and cache_lens [num_seqs] int64/int32/uint32.
    """
    return _call(_PAGED_ATTENTION, scale, _make_paged_attention, out, q, k_cache, v_cache, block_tables, cache_lens,
                 alibi_slopes)


def paged_attention_prefill(q, k_cache, v_cache, block_tables, seq_lens, cum_seq_lens_q, alibi_slopes=None,
                            scale: float = 1.0, *, out=None):
    """Causal attention of each sequence's run of new tokens over its paged K/V; returns ``out``.

    q [total_q_tokens, num_heads, head_size] holds the new tokens of all sequences back to back;
    seq_lens [num_seqs] are the total K/V lengths (history + new), cum_seq_lens_q [num_seqs + 1] the
    prefix sums of the new-token counts; both and block_tables share one index dtype.
    """
    return _call(_PAGED_ATTENTION_PREFILL, scale, _make_paged_attention_prefill, out, q, k_cache, v_cache, block_tables,
                 seq_lens, cum_seq_lens_q, alibi_slopes)


def paged_caching(k_cache, v_cache, k, v, slot_mapping):
    """Scatter ``k`` / ``v`` [num_tokens, num_kv_heads, d] into the pools in place; returns the pools."""
    _call(_PAGED_CACHING, 0, _make_paged_caching, k_cache, v_cache, k, v, slot_mapping)
    return k_cache, v_cache


def rope_paged_caching(k_cache, v_cache, k, v, slot_mapping, pos_ids, sin_table, cos_table,
                       algo: int = lib.RoPEAlgo.GPT_NEOX, *, q=None, q_out=None):
    """Rotate ``k`` [num_tokens, num_kv_heads, head_size] by the rows ``pos_ids`` of the sin / cos tables
    [table_len, head_size / 2] and scatter it, and ``v`` unchanged, into their slots of the paged pools, in one
    launch; returns the pools. The result of the reference's ``rope`` followed by ``paged_caching``
    (python/infinicore/ops/paged_caching.py:5-15 for the scatter's argument order). With ``q``
    [num_tokens, num_heads, head_size] the query is rotated in the same launch, into ``q_out`` (default: in
    place), and the call returns ``(k_cache, v_cache, q_out)``."""
    if q is not None:
        if q_out is None:
            q_out = q
        _call(_ROPE_QK_PAGED_CACHING, int(algo), _make_rope_qk_paged_caching, q_out, q, k_cache, v_cache, k, v, slot_mapping,
              pos_ids, sin_table, cos_table)
        return k_cache, v_cache, q_out
    _call(_ROPE_PAGED_CACHING, int(algo), _make_rope_paged_caching, k_cache, v_cache, k, v, slot_mapping, pos_ids, sin_table,
          cos_table)
    return k_cache, v_cache


def kv_caching(k_cache, v_cache, k, v, past_kv_lengths):
    """Append ``k`` / ``v`` [batch, num_kv_heads, seq_len, d] to the contiguous caches
    [batch, num_kv_heads, max_seq_len, d] behind the first ``past_kv_lengths[b]`` positions, in place; returns
    the caches (argument order of the reference's infiniopKVCaching, include/infiniop/ops/kv_caching.h:8-29)."""
    _call(_KV_CACHING, 0, _make_kv_caching, k_cache, v_cache, k, v, past_kv_lengths)
    return k_cache, v_cache
