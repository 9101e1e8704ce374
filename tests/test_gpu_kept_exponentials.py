"""Short batches whose exponentials the forward leaves in the memory-side cache for the backward (past_cache in csrc/lmhead.hip):
the contractions' order is that of the gradient's kind, and every saving forward keeps them. dWeight stored, added to a gradient
and written in bf16 leave the same accumulators, so they agree bit for bit (fp32 plus the old values, its rounding), and
dHidden does not depend on which of them ran in front of it. Elements against fp32 torch: |error| <= 2 % of the largest
magnitude, the bound of bf16 operands that test_gpu_dweight_chain.py states."""

import re

import pytest
import torch

from areal_amd.functional import fused_lm_head_logprobs_entropy

pytestmark = pytest.mark.gpu

V = 137984  # x 1024 hidden: 270 MiB of weight, more than the cache holds; 256 or 300 tokens: 67 or 101 MiB of exponentials
H = 1024


def _inputs(dev, T, V=V):
    g = torch.Generator(device=dev).manual_seed(T)
    hidden = torch.randn(T, H, generator=g, device=dev).bfloat16()
    weight = (torch.randn(V, H, generator=g, device=dev) * (2.0 / H ** 0.5)).bfloat16()
    return hidden, weight, torch.randint(0, V, (T,), generator=g, device=dev), torch.randn(T, generator=g, device=dev), g


def _backward(inputs, accum, *, frozen=False, **options):
    hidden, weight, labels, grad = inputs[:4]
    h, w = hidden.clone().requires_grad_(True), weight.clone().requires_grad_(not frozen)
    out = fused_lm_head_logprobs_entropy(h, w, labels, weight_grad_accum=accum, **options)
    out.logprobs.backward(grad)
    return (w.grad if accum is None else accum), h.grad, out


@pytest.mark.parametrize("kind", ["plain", "bias", "scale", "moments", "bias and moments"])
@pytest.mark.parametrize("T", [256, 300])
def test_three_outputs_of_dweight_agree(dev, T, kind):
    inputs = _inputs(dev, T)
    hidden, weight, labels, grad, g = inputs
    bias = torch.randn(V, generator=g, device=dev) if "bias" in kind else None
    options = dict(bias=bias, logit_scale=0.5 if kind == "scale" else 1.0, with_moments="moments" in kind, save_probs=True)
    before = torch.randn(V, H, generator=g, device=dev)
    plain, dh, out = _backward(inputs, torch.zeros(V, H, device=dev), **options)
    added, dh_added, _ = _backward(inputs, before.clone(), **options)
    half, dh_half, _ = _backward(inputs, None, **options)
    assert torch.equal(added, before + plain)
    assert torch.equal(half, plain.bfloat16())
    assert torch.equal(dh, dh_added) and torch.equal(dh, dh_half)

    h32, w32 = hidden.float(), weight.float()
    logits = (h32 @ w32.t()) * options["logit_scale"]
    if bias is not None:
        logits += bias
    logp = torch.log_softmax(logits, -1)
    own = torch.arange(T, device=dev)
    torch.testing.assert_close(out.logprobs.detach(), logp[own, labels], rtol=1e-5, atol=1e-4)
    torch.testing.assert_close(out.entropy, -(logp.exp() * logp).sum(-1), rtol=1e-4, atol=1e-4)
    if "moments" in kind:
        torch.testing.assert_close(out.vocab_mean_logits, logits.mean(-1), rtol=1e-4, atol=1e-4)
    d = -logp.exp()
    d[own, labels] += 1
    d *= grad[:, None] * options["logit_scale"]
    for got, want in ((plain, d.t() @ h32), (dh.float(), d @ w32)):
        assert (got - want).abs().max().item() <= 2e-2 * want.abs().max().item()


@pytest.mark.parametrize("kind", ["plain", "bias", "scale", "moments", "recompute"])
@pytest.mark.parametrize("gradient", ["bf16", "fp32"])
def test_order_and_hints(dev, gradient, kind):
    """Kernels of one backward in their order: an fp32 dWeight, which goes through the cache, behind dHidden, one in bf16,
    which goes past it, in front; a backward without saved exponentials always behind. The kernels' last template argument
    says whether they take part."""
    inputs = _inputs(dev, 300)
    options = dict(bias=torch.randn(V, device=dev) if kind == "bias" else None, logit_scale=0.5 if kind == "scale" else 1.0,
                   with_moments=kind == "moments", save_probs=kind != "recompute")
    accum = torch.zeros(V, H, device=dev) if gradient == "fp32" else None
    _backward(inputs, accum, **options)
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        _backward(inputs, accum, **options)
        torch.cuda.synchronize()
    events = sorted((e.time_range.start, e.name) for e in prof.events() if "gemm16_sweep<" in e.name)
    sweeps = [(int(re.search(r"gemm16_sweep<(\d)", n).group(1)), re.search(r"(true|false)\s*>", n).group(1) == "true", n) for _, n in events]
    first = {}
    for i, (variant, past, name) in enumerate(sweeps):
        first.setdefault(variant, (i, past, name))
    if kind == "recompute":  # 300 tokens are no whole k-tiles: dWeight reads a transposed copy (variant 0)
        assert first[2][1] is False, first
        return
    assert first[0][1] is True, first            # the forward keeps
    assert first[2][1] is True, first            # dHidden streams the weight
    assert first[1][1] is (gradient == "bf16"), first
    assert (first[1][0] < first[2][0]) is (gradient == "bf16"), first


@pytest.mark.parametrize("T, vocab, kept", [(256, V, True), (256, 131008, False), (129, V, True), (128, V, False), (128, 151936, True), (768, V, True),
                                            (896, 131136, False), (897, 131136, False)])
def test_sizes_that_keep(dev, T, vocab, kept):
    """A weight that fits the cache itself is not streamed (131008 x 1024), one that nearly does not for 128 tokens, and of many
    tokens or exponentials (224 MiB) nothing is kept."""
    inputs = _inputs(dev, T, vocab)
    _backward(inputs, None, save_probs=True)
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        _backward(inputs, None, save_probs=True)
        torch.cuda.synchronize()
    events = sorted((e.time_range.start, e.name) for e in prof.events() if "gemm16_sweep<" in e.name)
    past = {v: [re.search(r"(true|false)\s*>", n).group(1) == "true" for _, n in events if f"gemm16_sweep<{v}" in n][0] for v in (0, 1, 2)}
    assert past == {0: kept, 1: kept, 2: kept}


@pytest.mark.parametrize("T, gradient, saved, hint", [
    (256, None, True, False), (300, None, True, True), (256, None, False, False), (320, None, False, False),
    (256, "bf16", True, True), (256, "bf16", False, True), (300, "bf16", False, False), (640, "bf16", False, False),
    (256, "fp32", True, True), (256, "fp32", False, False), (640, "fp32", False, False)])
def test_weight_under_the_hint(dev, T, gradient, saved, hint):
    """Whether dHidden reads the weight past the cache: not of one tile of tokens alone (a weight without a gradient), and of dlogits made
    anew only next to a bf16 dWeight that reads them as they are written, of few tokens. Its values do not depend on it."""
    inputs = _inputs(dev, T)
    accum = torch.zeros(V, H, device=dev) if gradient == "fp32" else None
    _backward(inputs, accum, save_probs=saved, frozen=gradient is None)
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        _, dh, _ = _backward(inputs, accum, save_probs=saved, frozen=gradient is None)
        torch.cuda.synchronize()
    names = [e.name for e in prof.events() if "gemm16_sweep<2" in e.name]
    assert names and all(re.search(r"(true|false)\s*>", n).group(1) == str(hint).lower() for n in names), names
    hidden, weight, labels, grad, _ = inputs
    d = -torch.softmax(hidden.float() @ weight.float().t(), -1)
    d[torch.arange(T, device=dev), labels] += 1
    want = (d * grad[:, None]) @ weight.float()
    assert (dh.float() - want).abs().max().item() <= 2e-2 * want.abs().max().item()
