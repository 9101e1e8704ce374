"""Packing and padding of token batches on MI355X.

Same signatures and return structures as the reference's ``areal/utils/data.py``
``pack_tensor_dict`` (:496-545) and ``pad_packed_tensor_dict`` (:822-982), and the unpack ->
reorder -> pad-and-stack composition of ``reorder_and_pad_outputs``
(``areal/engine/core/train_engine.py:110-144``).  Every per-sequence Python loop of the
reference (one ``.item()`` or slice assignment per sequence and tensor) is one gather kernel by
``cu_seqlens`` here; a call waits for the GPU once (for the total length and the
longest sequence, which the reference returns as Python ints as well). What a call does around its
kernels is native (``csrc/host.cpp``).
"""

from __future__ import annotations

import ctypes
import itertools
import math
from typing import Any

import torch

from areal_amd import _lib

N_TOKENS_PER_PAGE = 256  # data.py:819


def _elem_bytes(t: torch.Tensor, lead_dims: int) -> int:
    return int(math.prod(t.shape[lead_dims:])) * t.element_size()


def _fill_bytes(dtype: torch.dtype, value: float):
    """Bit pattern of ``value`` in ``dtype`` as a ctypes buffer (<= 16 bytes)."""
    raw = _fill_pattern(dtype, value)
    return ctypes.create_string_buffer(raw, len(raw)), len(raw)


def _is_plain_zero(value) -> bool:
    return type(value) in (int, float) and value == 0 and math.copysign(1.0, value) > 0


def _fill_pattern(dtype: torch.dtype, value: float) -> bytes:
    if _is_plain_zero(value):
        return bytes(dtype.itemsize)  # zero is all zero bits in every type
    return torch.tensor([value], dtype=dtype).view(torch.uint8).numpy().tobytes()


def pack_tensor_dict(data: dict[str, Any]) -> dict[str, Any]:
    """Pack a dict of ``[B, S, ...]`` tensors into ``[total_length, ...]``; ``attention_mask`` is
    replaced by ``cu_seqlens`` (int32 ``[B+1]``) and ``max_seqlen`` (int)."""
    assert "attention_mask" in data, "Input data must contain 'attention_mask' key."
    attention_mask = data["attention_mask"]
    assert attention_mask.ndim == 2, "Attention mask must be a 2D tensor."
    if type(data) is not dict:
        data = dict(data)
    return _lib.host().pack_dict(data, attention_mask)


def _realign(lib, dev, value, cu_old, n_old, cu_new, n_new, total_new, pad_value, position_ids, whole_arange):
    out_shape = (total_new, *value.shape[1:])
    out = torch.empty(out_shape, dtype=value.dtype, device=value.device)
    src = value.contiguous()
    if position_ids:
        if value.dtype != torch.int64:
            src = src.to(torch.int64)
            out = torch.empty(out_shape, dtype=torch.int64, device=value.device)
        fill, nfill = None, 0
    else:
        fill, nfill = _fill_bytes(value.dtype, pad_value)
    rc = lib.areal_realign_packed(
        _lib.ptr(None if whole_arange else src), _lib.ptr(out), _lib.ptr(cu_old), n_old,
        _lib.ptr(cu_new), n_new, _elem_bytes(src, 1), fill, nfill, int(position_ids), total_new,
        _lib.stream_ptr(dev),
    )
    _lib.check(rc, "areal_realign_packed")
    return out.to(value.dtype) if out.dtype != value.dtype else out


def pad_packed_tensor_dict(
    data: dict[str, Any],
    pad_to_length: int,
    pad_value: float = 0.0,
    seq_align_to: int | None = None,
) -> tuple[dict[str, Any], int, torch.Tensor, int | None]:
    """Pad a packed dict of tensors to ``pad_to_length`` by appending one pad sequence, after
    optionally aligning every sequence to a multiple of ``seq_align_to``.  Returns
    ``(padded_data, pad_length, old_cu_seqlens, align_to_length)``."""
    assert "cu_seqlens" in data, "Input data must contain 'cu_seqlens' key."
    assert "max_seqlen" in data, "Input data must contain 'max_seqlen' key."
    lib = _lib.load()
    cu_seqlens = data["cu_seqlens"]
    dev = _lib.require_gpu(cu_seqlens)
    cu_seqlens = cu_seqlens.to(torch.int32).contiguous()
    max_seqlen = data["max_seqlen"]
    n_seqs = cu_seqlens.numel() - 1
    align_to_length = None
    if seq_align_to is not None:
        old_cu_seqlens = cu_seqlens.clone()
        input_lens = cu_seqlens[1:] - cu_seqlens[:-1]
        lens_padded = input_lens + (-input_lens) % seq_align_to
        cu_padded = torch.zeros(n_seqs + 1, dtype=torch.int32, device=dev)
        cu_padded[1:] = torch.cumsum(lens_padded, dim=0)
        total_length, total_padded, max_padded = torch.stack(
            [cu_seqlens[-1], cu_padded[-1], lens_padded.max()]
        ).tolist()
    else:
        # The total is on the device, behind what the stream holds (the packing itself, as a rule). The padding is launched
        # for the total that the tensors' shapes suggest and reports the one it met: the host prepares it while the
        # GPU packs (25.3 -> 18.0 us of a batch of 256 x 4096).
        total_length = None
        if type(data) is dict and type(pad_to_length) is int and _is_plain_zero(pad_value):
            padded = _lib.host().pad_likely(data, cu_seqlens, pad_to_length)
            if type(padded) is tuple:
                return (*padded, None)
            total_length = padded
        if total_length is None:
            total_length = _lib.host().LastValue(cu_seqlens).wait()

    if seq_align_to is not None:
        aligned: dict[str, Any] = {}
        for key, value in data.items():
            if key == "cu_seqlens":
                aligned[key] = cu_padded
            elif key == "max_seqlen":
                aligned[key] = max_padded
            elif key == "position_ids":
                three = value.ndim == 2 and value.shape[1] == 3
                aligned[key] = _realign(lib, dev, value, cu_seqlens, n_seqs, cu_padded, n_seqs, total_padded,
                                        0.0, True, whole_arange=not three)
            elif _is_token_tensor(key, value, total_length):
                aligned[key] = _realign(lib, dev, value.reshape(total_length), cu_seqlens, n_seqs, cu_padded,
                                        n_seqs, total_padded, pad_value, False, False)
            else:
                aligned[key] = value
        data = aligned
        align_to_length = total_padded
        lcm = math.lcm(seq_align_to, N_TOKENS_PER_PAGE)
        pad_to_length = (pad_to_length + lcm - 1) // lcm * lcm
        cu_seqlens, max_seqlen, total_length = cu_padded, max_padded, total_padded
        if pad_to_length < total_length:
            pad_to_length = (total_length + lcm - 1) // lcm * lcm

    pad_length = pad_to_length - total_length
    if pad_length < 0:
        raise ValueError(f"pad_to_length {pad_to_length} is smaller than total length {total_length}.")
    if pad_length == 0:
        return data, pad_length, cu_seqlens.clone() if seq_align_to is None else old_cu_seqlens, align_to_length
    padded, cu_copy = _with_pad_sequence(lib, dev, data, cu_seqlens, total_length, pad_to_length, pad_value)
    return padded, pad_length, cu_copy if seq_align_to is None else old_cu_seqlens, align_to_length


def _is_token_tensor(key, value, total):
    if key == "position_ids":
        return torch.is_tensor(value)
    return torch.is_tensor(value) and value.numel() == total


def _with_pad_sequence(lib, dev, data, cu_seqlens, total_length, pad_to_length, pad_value):
    """One more sequence behind the others, and a copy of the offsets before it: eight tensors per launch, the first of
    which also writes the two offset arrays."""
    max_seqlen = data["max_seqlen"]
    n_seqs = cu_seqlens.numel() - 1
    new_cu = torch.empty(n_seqs + 2, dtype=torch.int32, device=dev)
    cu_copy = torch.empty_like(cu_seqlens)
    padded: dict[str, Any] = {}
    moved, sources, patterns = [], [], []  # keys of the tensors that are copied, what is copied, its fill
    fills: dict[torch.dtype, bytes] = {}
    for key, value in data.items():
        if key == "cu_seqlens":
            padded[key] = new_cu
        elif key == "max_seqlen":
            padded[key] = max(max_seqlen, pad_to_length - total_length)
        elif not _is_token_tensor(key, value, total_length):
            padded[key] = value
        elif key == "position_ids" and (value.dtype != torch.int64 or value.shape[:1] != (total_length,)):
            padded[key] = _realign(lib, dev, value, cu_seqlens, n_seqs, _batch_pad(cu_seqlens, pad_to_length),
                                   n_seqs + 1, pad_to_length, 0.0, True, False)
        else:
            padded[key] = value
            moved.append(key)
            if key == "position_ids":  # they go on from 0
                sources.append(value)
                patterns.append(b"")
                continue
            sources.append(value.reshape(total_length))
            if value.dtype not in fills:
                fills[value.dtype] = _fill_pattern(value.dtype, pad_value)
            patterns.append(fills[value.dtype])
    outs = _lib.host().pad_rows(sources, patterns, cu_seqlens, cu_copy, new_cu, total_length, pad_to_length)
    padded.update(zip(moved, outs))
    return padded, cu_copy


def _batch_pad(cu_seqlens, pad_to_length):
    return torch.nn.functional.pad(cu_seqlens, (0, 1), value=pad_to_length)


def unpack_reorder_pad(
    packed: torch.Tensor,
    seqlens: list[int],
    backward_indices: list[int] | None = None,
) -> torch.Tensor:
    """``pad_and_stack_tensors_along_first_dim(reorder_list(unpack_sequence(packed, lens=seqlens),
    backward_indices))`` in one gather: row ``r`` of the ``[n, max(seqlens), ...]`` result holds
    packed sequence ``backward_indices[r]``, zero padded."""
    lib = _lib.load()
    dev = _lib.require_gpu(packed)
    if type(seqlens) is list and (backward_indices is None or type(backward_indices) is list):
        out = _lib.host().unpack_rows(packed, seqlens, backward_indices)
        if out is not None:
            return out
    n = len(seqlens)
    if backward_indices is not None:
        assert len(set(backward_indices)) == n
    if sum(seqlens) != packed.shape[0]:
        raise ValueError(f"seqlens sum to {sum(seqlens)}, the packed tensor has {packed.shape[0]} rows")
    # the offsets and the order travel in one copy
    order = backward_indices if backward_indices is not None else ()
    table = torch.tensor([0, *itertools.accumulate(seqlens), *order], dtype=torch.int32).to(dev)
    cu = table[: n + 1]
    row_seq = table[n + 1 :] if backward_indices is not None else None
    max_len = max(seqlens) if n > 0 else 0
    src = packed.contiguous()
    out = torch.empty((n, max_len, *packed.shape[1:]), dtype=packed.dtype, device=dev)
    rc = lib.areal_unpack_to_padded(
        _lib.ptr(src), _lib.ptr(out), _lib.ptr(cu), _lib.ptr(row_seq), n, max_len,
        _elem_bytes(src, 1), None, 0, _lib.stream_ptr(dev),
    )
    _lib.check(rc, "areal_unpack_to_padded")
    return out


def reorder_and_pad_outputs(outputs, output_seqlens, mb_list, aggregate_fn=torch.cat) -> torch.Tensor:
    """Aggregate micro-batch outputs, then unpack / reorder / pad in one kernel
    (``train_engine.py:110-144``).  ``mb_list`` needs ``forward_indices`` and ``backward_indices``."""
    res = aggregate_fn(outputs)
    seqlens = [output_seqlens[i] for i in mb_list.forward_indices]
    return unpack_reorder_pad(res, seqlens, list(mb_list.backward_indices))
