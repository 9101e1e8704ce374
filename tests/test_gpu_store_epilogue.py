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
