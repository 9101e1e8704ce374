"""The fp32 gradient of a master weight that has none when the forward runs: it is looked up when the backward
runs, so whatever is there by then is added to. Against the gradient that a given accumulator receives."""

import functools
from types import SimpleNamespace

import pytest
import torch

from areal_amd.engine import FusedLMHeadAdapter
from areal_amd.functional import fused_lm_head_logprobs_entropy
from areal_amd.functional.lm_head import _lm_head

pytestmark = pytest.mark.gpu

T, H, V = 320, 128, 1536


def _parts(dev, n, t=T, v=V):
    g = torch.Generator().manual_seed(t)
    param = torch.nn.Parameter((torch.randn(v, H, generator=g) * 0.1).to(dev))
    weight = param.detach().bfloat16()
    parts = [(torch.randn(t, H, generator=g).bfloat16().to(dev).requires_grad_(True),
              torch.randint(0, v, (t,), generator=g).to(dev), torch.randn(t, generator=g).to(dev)) for _ in range(n)]
    return param, weight, parts


def _forward(param, weight, part, save_probs=True):
    hidden, labels, _ = part
    return _lm_head(hidden, weight, labels, 1.0, 1.0, None, None, save_probs, False, None, param).logprobs


def _want(weight, parts):
    accum = torch.zeros(weight.shape, device=weight.device)
    for hidden, labels, g in parts:
        out = fused_lm_head_logprobs_entropy(hidden.detach().requires_grad_(True), weight, labels, save_probs=True,
                                             weight_grad_accum=accum)
        out.logprobs.backward(g)
    return accum


def test_two_forwards_before_either_backward(dev):
    param, weight, parts = _parts(dev, 2)
    outs = [_forward(param, weight, p) for p in parts]
    assert param.grad is None
    for out, p in zip(outs, parts):
        out.backward(p[2])
    assert torch.equal(param.grad, _want(weight, parts))


@pytest.mark.parametrize("strides", ["contiguous", "transposed", "expanded rows"])
def test_gradient_set_between_forward_and_backward(dev, strides):
    param, weight, parts = _parts(dev, 1)
    out = _forward(param, weight, parts[0])
    before = torch.randn(V, H, device=dev)
    if strides == "transposed":
        before = before.t().contiguous().t()
    elif strides == "expanded rows":
        before = torch.randn(V, 2 * H, device=dev)[:, :H]
    param.grad = before
    start = before.clone()
    out.backward(parts[0][2])
    assert param.grad is before and param.grad.stride() == before.stride()
    # one fp32 addition per element in either order
    torch.testing.assert_close(param.grad, start + _want(weight, parts), rtol=2e-7, atol=2e-7 * start.abs().max().item())


@pytest.mark.parametrize("have_grad", [False, True])
def test_batch_without_any_loss_leaves_a_gradient_of_zeros(dev, have_grad):
    """No loss of the batch reaches the weight: its gradient is zeros, or what it was."""
    param, _, parts = _parts(dev, 2)
    lm = SimpleNamespace(model=lambda hidden: hidden, lm_head=SimpleNamespace(weight=param, bias=None))
    if have_grad:
        param.grad = torch.ones_like(param)
    micro = [dict(model_inputs=dict(hidden=h), mb_input=dict(labels=y)) for h, y, _ in parts]
    adapter = FusedLMHeadAdapter(lm)
    adapter._scaled_loss = lambda inputs, *args: inputs["hidden"].float().sum()
    adapter.forward_backward_batch(micro, functools.partial(lambda: None), lambda mb: 1.0)
    assert torch.equal(param.grad, torch.ones_like(param) if have_grad else torch.zeros_like(param))


def test_failing_backward_sets_no_gradient(dev):
    """The backward's workspace does not fit: the error leaves no half-made gradient for a smaller batch to be
    added to."""
    param, weight, parts = _parts(dev, 1, t=4096, v=16384)
    out = _forward(param, weight, parts[0], save_probs=False)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # room for the gradient (8 MiB), not for the 128 MiB of dlogits
    room = torch.cuda.memory_reserved(dev) + (64 << 20)
    torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(dev).total_memory, dev)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            out.backward(parts[0][2], retain_graph=True)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
    assert param.grad is None
    out.backward(parts[0][2])
    want = torch.zeros_like(param)
    again = fused_lm_head_logprobs_entropy(parts[0][0], weight, parts[0][1], save_probs=False, weight_grad_accum=want)
    again.logprobs.backward(parts[0][2])
    assert torch.equal(param.grad, want)
