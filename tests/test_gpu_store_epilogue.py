"""The store epilogues of the hand-scheduled contraction where whole and partial 128 x 128 sub-tiles of a wave meet in
one launch: hidden sizes that end 8, 64, 72 and 128 columns into a sub-tile (and 224-wide tiles), vocabularies and token
counts that end inside one. dWeight added to a gradient, and written in bf16, has to be bit for bit the fp32 result
plus the old values, and its rounding: the three leave the accumulators by different routes. Elements against fp32
torch: |error| <= 2 % of the largest magnitude, the bound of bf16 operands that test_gpu_dweight_chain.py states."""

import pytest
import torch

from areal_amd.functional import fused_lm_head_logprobs_entropy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,V", [(130, 264, 640), (257, 320, 832), (200, 456, 4160), (384, 896, 1088), (509, 640, 16960)])
def test_three_outputs_of_dweight_agree(dev, T, H, V):
    g = torch.Generator(device=dev).manual_seed(T * 7 + H + V)
    hidden = torch.randn(T, H, generator=g, device=dev).bfloat16()
    weight = (torch.randn(V, H, generator=g, device=dev) * (2.0 / H ** 0.5)).bfloat16()
    labels = torch.randint(0, V, (T,), generator=g, device=dev)
    grad = torch.randn(T, generator=g, device=dev)
    before = torch.randn(V, H, generator=g, device=dev)

    def backward(accum):
        h, w = hidden.clone().requires_grad_(True), weight.clone().requires_grad_(True)
        out = fused_lm_head_logprobs_entropy(h, w, labels, save_probs=True, weight_grad_accum=accum)
        out.logprobs.backward(grad)
        return (w.grad if accum is None else accum), h.grad

    plain, dh = backward(torch.zeros(V, H, device=dev))
    added, dh_added = backward(before.clone())
    half, dh_half = backward(None)
    assert torch.equal(added, before + plain)
    assert torch.equal(half, plain.bfloat16())
    assert torch.equal(dh, dh_added) and torch.equal(dh, dh_half)

    h32, w32 = hidden.float(), weight.float()
    d = -torch.softmax(h32 @ w32.t(), -1)
    d[torch.arange(T, device=dev), labels] += 1
    d *= grad[:, None]
    for got, want in ((plain, d.t() @ h32), (dh.float(), d @ w32)):
        assert (got - want).abs().max().item() <= 2e-2 * want.abs().max().item()


# either side of the rule on keeping the exponentials in the memory-side cache (768 tokens of this vocabulary), 224-wide and
# whole tiles, a bias (another forward epilogue), a vocabulary that is no multiple of 64 (the transposed weight)
@pytest.mark.parametrize("T,H,V,bias", [(130, 896, 151936, False), (768, 896, 151936, False), (769, 896, 151936, False),
                                        (509, 1024, 128256, False), (200, 1024, 128256, True), (200, 1024, 128250, False)])
def test_exponentials_kept_for_the_backward(dev, T, H, V, bias):
    g = torch.Generator(device=dev).manual_seed(T + H + V)
    hidden = torch.randn(T, H, generator=g, device=dev).bfloat16().requires_grad_(True)
    weight = (torch.randn(V, H, generator=g, device=dev) * (2.0 / H ** 0.5)).bfloat16().requires_grad_(True)
    b = torch.randn(V, generator=g, device=dev) if bias else None
    labels = torch.randint(0, V, (T,), generator=g, device=dev)
    grad = torch.randn(T, generator=g, device=dev)
    out = fused_lm_head_logprobs_entropy(hidden, weight, labels, bias=b, save_probs=True)
    out.logprobs.backward(grad)
    h32, w32 = hidden.detach().float(), weight.detach().float()
    logits = h32 @ w32.t()
    if bias:
        logits += b
    logp = torch.log_softmax(logits, -1)
    own = torch.arange(T, device=dev)
    torch.testing.assert_close(out.logprobs.detach(), logp[own, labels], rtol=1e-5, atol=1e-4)
    d = -logp.exp()
    del logits, logp
    d[own, labels] += 1
    d *= grad[:, None]
    for got, want in ((weight.grad, d.t() @ h32), (hidden.grad, d @ w32)):
        assert (got.float() - want).abs().max().item() <= 2e-2 * want.abs().max().item()
