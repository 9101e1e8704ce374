"""``gather_logprobs`` / ``gather_logprobs_entropy`` with the reference's signatures
(``areal/utils/functional/vocab_parallel.py:564-651``), computed by one pass of the row
kernels in ``csrc/logits_rows.hip`` over materialised logits.

``chunk_size`` is accepted and ignored: the reference chunks rows to bound the fp32 copy of
the logits (``:42-62``); the kernel never makes that copy. The autograd node is native
(``csrc/host.cpp``).  ``tp_group`` with more than one
rank is outside the one-GPU scope and raises.
"""

from __future__ import annotations

import math

import torch
import torch.distributed as dist

from areal_amd import _lib

def _validate(logits, labels, temperature, tp_group):
    if tp_group is not None and dist.is_initialized() and dist.get_world_size(tp_group) > 1:
        raise NotImplementedError("vocab-parallel logits over several GPUs are not built here")
    if not math.isfinite(temperature) or temperature <= 0:
        raise ValueError(f"temperature must be positive, got {temperature}")
    if tuple(logits.shape[:-1]) != tuple(labels.shape):
        raise ValueError(
            "logits leading dimensions must match labels: "
            f"got {tuple(logits.shape)} and {tuple(labels.shape)}"
        )
    assert logits.numel() > 0, "Input logits must have at least one element"


def gather_logprobs(
    logits: torch.Tensor,
    labels: torch.Tensor,
    temperature: float = 1.0,
    tp_group=None,
    chunk_size: int = 1024,
) -> torch.Tensor:
    """``log_softmax(logits.float() / temperature)[labels]`` with shape ``labels.shape``."""
    del chunk_size
    _validate(logits, labels, temperature, tp_group)
    return _lib.host().logits_logprobs(logits, labels, temperature, False)[0]


def gather_logprobs_entropy(
    logits: torch.Tensor,
    labels: torch.Tensor,
    temperature: float = 1.0,
    tp_group=None,
    chunk_size: int = 1024,
    reuse_logits: bool = False,
) -> tuple[torch.Tensor, torch.Tensor]:
    """Label log-probabilities and softmax entropy in one pass; both are differentiable,
    as on the reference's single-GPU path (``vocab_parallel.py:75-82``).

    ``reuse_logits`` asks the reference to overwrite fp32 logits in place and lets it fall back
    to the regular path otherwise (``:625-640``); this implementation needs no fp32 copy, so the
    regular path is always taken.
    """
    del chunk_size, reuse_logits
    _validate(logits, labels, temperature, tp_group)
    return tuple(_lib.host().logits_logprobs(logits, labels, temperature, True))
