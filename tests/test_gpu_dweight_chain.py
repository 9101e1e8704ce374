"""dWeight launches of more tiles than the chip has CUs: a workgroup then takes several of them, the next
one's operands arriving while this one is stored. Ragged last tiles of either operand (fetched through a
window that ends with the operand), 256- and 224-wide tiles, an operand of one tile, an odd number of
k-tiles, and a hidden size that the chain does not take (not a multiple of 16). The last four lie either side of the
rule on 8 tiles of hidden size and 8192 tokens, beyond which the tiles are laid out in super-blocks instead.

Every element is compared with fp32 torch: |error| <= 2 % of the gradient's largest magnitude, the bound of
bf16 operands and outputs that the elementwise test of the tile widths uses."""

import pytest
import torch

from areal_amd.functional import fused_lm_head_logprobs_entropy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["saved", "recompute", "fp32", "fp32_accumulate"])
@pytest.mark.parametrize("T,H,V", [
    (130, 1056, 16448), (256, 1792, 12992), (192, 2496, 16384), (128, 520, 32768), (200, 128, 70000), (320, 256, 140032),
    (8192, 2056, 9000), (8320, 2048, 9000), (8320, 2056, 9000), (8320, 2304, 8192),
])
def test_every_element_of_a_chain(dev, T, H, V, mode):
    g = torch.Generator(device=dev).manual_seed(T + H + V)
    hidden = torch.randn(T, H, generator=g, device=dev).bfloat16().requires_grad_(True)
    weight = (torch.randn(V, H, generator=g, device=dev) * (2.0 / H ** 0.5)).bfloat16().requires_grad_(True)
    labels = torch.randint(0, V, (T,), generator=g, device=dev)
    grad = torch.randn(T, generator=g, device=dev)
    start = 0.25 if mode == "fp32_accumulate" else 0.0
    accum = torch.full((V, H), start, device=dev) if mode.startswith("fp32") else None
    out = fused_lm_head_logprobs_entropy(hidden, weight, labels, save_probs=mode != "recompute", weight_grad_accum=accum)
    out.logprobs.backward(grad)
    got = accum - start if accum is not None else weight.grad.float()

    h32, w32 = hidden.detach().float(), weight.detach().float()
    d = -torch.softmax(h32 @ w32.t(), -1)
    d[torch.arange(T, device=dev), labels] += 1
    want = (d * grad[:, None]).t() @ h32
    assert (got - want).abs().max().item() <= 2e-2 * want.abs().max().item()
