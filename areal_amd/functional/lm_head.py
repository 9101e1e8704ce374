"""Fused lm_head -> log-softmax -> label log-prob + entropy on MI355X.

Host-side counterpart of the reference's chunked LM head
(``areal/models/mcore/vocab_parallel_head.py:560-938`` and its wrapper
``chunked_lm_head_logprobs_entropy`` at ``:941-982``): same outputs
(``ChunkedLMHeadOutput``), same error behaviour.  The arithmetic runs in the HIP kernels of
``csrc/lmhead.hip`` through the C ABI, allocation and the autograd node in ``csrc/host.cpp``.

Two ways of carrying state to the backward:

* ``save_probs=False``: what the reference does -- row max and sum of exponentials per token,
  never a ``[T, V]`` tensor; the backward recomputes the logits chunk by chunk
  (``vocab_parallel_head.py:806-829``).
* ``save_probs=True``: the forward also writes the softmax exponentials as a bf16 ``[T, V]``
  tensor (2 bytes per logit), relative to a per-row reference estimated before the sweep; the
  backward contracts that buffer as it is (the per-row factor of dlogits goes to the output
  rows of dHidden and to the hidden states for dWeight) and skips the recomputation, a quarter
  of the step's matrix work.  The reference's logits-in path saves the same amount through
  autograd; 288 GB of HBM make it the default while it fits ``SAVE_PROBS_BYTES_LIMIT`` and
  60 % of the memory still available.  If some row's maximum logit lies more than 100 binades
  (69 nats at temperature 1) above its estimate, the kernel reports it, repeats the sweep
  without saving on the device (so the outputs are right without a host round trip), and the
  backward recomputes instead.
"""

from __future__ import annotations

import math
from typing import NamedTuple

import torch

from areal_amd import _lib

# Default budget for the backward workspace (bf16 dlogits of one token chunk in two layouts,
# plus transposed operands).  An MI355X has 288 GB of HBM, so one chunk normally covers the
# whole micro-batch.
DEFAULT_BWD_WORKSPACE_BYTES = 24 << 30

# save_probs=None keeps the exponentials when the bf16 [T, V] buffer is at most this large.
SAVE_PROBS_BYTES_LIMIT = 40 << 30


class ChunkedLMHeadOutput(NamedTuple):
    """Per-token outputs produced without materialising ``[T, V]`` logits.

    Field names and order follow ``vocab_parallel_head.py:497-506``.
    """

    logprobs: torch.Tensor
    entropy: torch.Tensor
    vocab_min_logits: torch.Tensor
    vocab_max_logits: torch.Tensor
    vocab_mean_logits: torch.Tensor
    vocab_norm_logits: torch.Tensor


def default_token_chunk(T: int, H: int, V: int, budget: int = DEFAULT_BWD_WORKSPACE_BYTES) -> int:
    """Largest token chunk (multiple of 256) whose backward workspace fits ``budget``."""
    return _lib.host().default_token_chunk(T, H, V, budget)


class _FusedLMHead(torch.autograd.Function):
    """The autograd node; its two directions are native (``lm_head`` and ``lm_head_backward`` of
    ``csrc/host.cpp``).  ``probs``, ``probs_ref`` and ``probs_status`` are the saved exponentials,
    their row references and whether they are usable, while the node holds them: plain
    attributes, not saved tensors, because the backward rewrites entries of ``probs`` in place."""

    @staticmethod
    def forward(ctx, hidden, weight, bias, labels, args):
        # args: a tuple, so that the accumulator and its owner in it are no inputs of the node. The
        # caller has ruled out no_grad mode.
        accum, owner = args[5:7]
        needs_grad = any(ctx.needs_input_grad[:2]) or accum is not None or owner is not None
        outs, saved, state = _lib.host().lm_head(hidden, weight, bias, labels, *args, True, needs_grad, False)
        ctx.save_for_backward(*saved)
        ctx.state = state
        ctx.probs, ctx.probs_ref, ctx.probs_status = state.probs, state.probs_ref, state.probs_status
        ctx.set_materialize_grads(False)
        ctx.mark_non_differentiable(*[o for o in outs[1:] if o is not None])
        return outs

    @staticmethod
    def backward(ctx, grad_logprobs, *unused):
        if grad_logprobs is None:
            return (None,) * 5
        ctx.probs = ctx.probs_ref = ctx.probs_status = None  # consumed; a second backward recomputes
        grads = _lib.host().lm_head_backward(ctx.state, ctx.saved_tensors, grad_logprobs, *ctx.needs_input_grad[:3])
        return (*grads, None, None)


def fused_lm_head_logprobs_entropy(
    hidden: torch.Tensor,
    weight: torch.Tensor,
    labels: torch.Tensor,
    *,
    temperature: float = 1.0,
    vocab_chunk: int | None = None,
    logit_scale: float = 1.0,
    bias: torch.Tensor | None = None,
    token_chunk: int | None = None,
    save_probs: bool | None = None,
    with_moments: bool = False,
    weight_grad_accum: torch.Tensor | None = None,
) -> ChunkedLMHeadOutput:
    """Label log-probabilities, entropy and vocabulary statistics of ``hidden @ weight.T``.

    Args:
        hidden: ``[..., H]`` bf16 final hidden states (packed tokens).
        weight: ``[V, H]`` bf16 lm_head weight (row = vocabulary id).
        labels: ``[...]`` integer labels, leading dimensions matching ``hidden``.
        temperature: softmax temperature (> 0).
        vocab_chunk: accepted for signature compatibility; the kernel sweeps the vocabulary
            in 256-row tiles whatever its value.
        logit_scale: multiplier applied to the logits before the softmax (> 0).
        bias: optional ``[V]`` bias added to the logits.
        token_chunk: tokens per backward chunk (bounds the bf16 dlogits workspace);
            ``None`` picks the largest chunk within ``DEFAULT_BWD_WORKSPACE_BYTES``.
        save_probs: keep the bf16 softmax exponentials for the backward instead of recomputing
            the logits; ``None`` decides by ``SAVE_PROBS_BYTES_LIMIT``.
        with_moments: also return ``vocab_mean_logits`` and ``vocab_norm_logits`` (two more
            operations per logit in the sweep); without it those two fields are ``None``.
        weight_grad_accum: an fp32 ``[V, H]`` tensor (normally the ``.grad`` of an fp32 master
            copy of ``weight``) that the weight gradient is ADDED to by the dWeight contraction
            itself, as Megatron's fp32 ``main_grad`` accumulation does
            (``vocab_parallel_head.py:873-879``); no gradient is then returned for ``weight``.
            The bias gradient, if any, is added in the same way only through autograd.

    Gradient flows through ``logprobs`` only (to ``hidden`` and ``weight``), as in the
    reference (``vocab_parallel_head.py:732-734``).
    """
    del vocab_chunk
    return _lm_head(
        hidden, weight, labels, temperature, logit_scale, bias, token_chunk, save_probs, with_moments,
        weight_grad_accum, None,
    )


def _lm_head(
    hidden, weight, labels, temperature, logit_scale, bias, token_chunk, save_probs, with_moments,
    weight_grad_accum, weight_grad_owner, logprobs_only=False,
) -> ChunkedLMHeadOutput:
    """``weight_grad_owner``: the fp32 parameter ``weight`` is a compute copy of; the weight gradient
    is added to its ``.grad`` as it is when the backward runs, or becomes it.
    ``logprobs_only`` (in no_grad mode): the other outputs are ``None`` and the sweep does not compute them."""
    if not math.isfinite(temperature) or temperature <= 0:
        raise ValueError(f"temperature must be positive, got {temperature}")
    if not math.isfinite(logit_scale) or logit_scale <= 0:
        raise ValueError(f"logit_scale must be positive, got {logit_scale}")
    if token_chunk is not None and token_chunk <= 0:
        raise ValueError(f"chunk_size must be positive, got {token_chunk}")
    if hidden.dtype != weight.dtype:
        raise ValueError(
            "chunked LM Head requires matching hidden and weight dtypes, got "
            f"{hidden.dtype} and {weight.dtype}"
        )
    if weight.ndim != 2 or hidden.size(-1) != weight.size(1):
        raise ValueError(
            f"weight must be [V, H] with H == hidden.size(-1); got {tuple(weight.shape)} "
            f"and {tuple(hidden.shape)}"
        )
    if hidden.numel() // max(hidden.size(-1), 1) != labels.numel():
        raise ValueError(
            "LM Head hidden leading dimensions must match labels: "
            f"got {tuple(hidden.shape)} and {tuple(labels.shape)}"
        )
    if hidden.dtype != torch.bfloat16:
        raise ValueError(f"the fused LM head computes in bf16; got {hidden.dtype}")
    if hidden.size(-1) % 8 != 0:
        raise ValueError(f"hidden size must be a multiple of 8, got {hidden.size(-1)}")
    if bias is not None and bias.shape != (weight.size(0),):
        raise ValueError(f"bias must have shape ({weight.size(0)},), got {tuple(bias.shape)}")
    if weight_grad_accum is not None:
        if weight_grad_accum.dtype != torch.float32 or weight_grad_accum.shape != weight.shape:
            raise ValueError(
                "weight_grad_accum must be an fp32 tensor of the weight's shape, got "
                f"{weight_grad_accum.dtype} {tuple(weight_grad_accum.shape)}"
            )
        if not weight_grad_accum.is_contiguous():
            raise ValueError("weight_grad_accum must be contiguous")
    if not torch.is_grad_enabled():
        save_probs = False  # no backward will come: keep nothing
        weight_grad_accum = weight_grad_owner = None
    args = (
        temperature, logit_scale, token_chunk or 0, -1 if save_probs is None else int(save_probs), with_moments,
        weight_grad_accum, weight_grad_owner, SAVE_PROBS_BYTES_LIMIT, DEFAULT_BWD_WORKSPACE_BYTES,
    )
    if torch.is_grad_enabled():
        values = _FusedLMHead.apply(hidden, weight, bias, labels, args)
    else:
        values = _lib.host().lm_head(hidden, weight, bias, labels, *args, False, False, logprobs_only)
    return ChunkedLMHeadOutput(*values)


def chunked_lm_head_logprobs_entropy(
    output_layer,
    hidden_states: torch.Tensor,
    weight: torch.Tensor,
    labels: torch.Tensor,
    *,
    temperature: float,
    chunk_size: int,
    logit_scale: float = 1.0,
) -> ChunkedLMHeadOutput:
    """The reference's entry point of the same name (``vocab_parallel_head.py:941-982``), for
    callers that hold an output layer object: the bias comes from ``output_layer.bias`` unless
    ``output_layer.skip_bias_add`` is set, ``chunk_size`` is validated and otherwise unused (the
    kernels hold no fp32 logits, so there is nothing to bound by it), and the layer options the
    fused path cannot honour are refused with the reference's errors. Tensor-parallel layers (a ``tp_group`` of more than one rank) are
    outside the one-GPU scope."""
    if not getattr(output_layer, "chunked_loss_supported", True):
        raise NotImplementedError(
            "chunked LM Head loss does not support this output-layer forward override"
        )
    config = getattr(output_layer, "config", None)
    if getattr(config, "defer_embedding_wgrad_compute", False):
        raise NotImplementedError(
            "chunked LM Head loss is incompatible with defer_embedding_wgrad_compute"
        )
    if getattr(output_layer, "gather_output", False):
        raise NotImplementedError(
            "chunked LM Head loss requires vocab-parallel (ungathered) output"
        )
    tp_group = getattr(output_layer, "tp_group", None)
    if tp_group is not None:
        import torch.distributed as dist

        if dist.is_initialized() and dist.get_world_size(tp_group) > 1:
            raise NotImplementedError("vocab-parallel LM heads over several GPUs are not built here")
    bias = None
    if not getattr(output_layer, "skip_bias_add", False):
        bias = getattr(output_layer, "bias", None)
    if chunk_size <= 0:
        raise ValueError(f"chunk_size must be positive, got {chunk_size}")
    return fused_lm_head_logprobs_entropy(
        hidden_states, weight, labels, temperature=temperature, logit_scale=logit_scale, bias=bias,
        with_moments=True,
    )

