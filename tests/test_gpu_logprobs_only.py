"""Forward-only label log-probabilities, whose sweep sums relative to a reference taken from a token's first
logits: ragged token counts and vocabularies (a last tile that overlaps its predecessor, one in a launch of its
own), odd contraction lengths, and rows whose logits rise above the reference by more than the window, once and again
from tile to tile, lie far below zero, or are not finite.

Against float64 torch on the same bf16 operands. The kernel's logits are fp32 sums of H products, its sum of exponentials one of
fp32 terms of one sign: |error| <= 2^-20 of the largest |logit| + 2^-18."""

import pytest
import torch

from areal_amd.engine import FusedLMHeadAdapter, compute_logprobs
from areal_amd.functional import fused_lm_head_logprobs_entropy

pytestmark = pytest.mark.gpu


def _want(hidden, weight, labels, temperature=1.0, bias=None):
    x = hidden.double() @ weight.double().t()
    x = (x if bias is None else x + bias.double()) / temperature
    ok = (labels >= 0) & (labels < weight.size(0))
    own = torch.where(ok, x.gather(1, labels.clamp(0, weight.size(0) - 1)[:, None])[:, 0], 0.0)
    return own - torch.logsumexp(x, -1), 2.0 ** -20 * x.abs().max().item() + 2.0 ** -18


@pytest.mark.parametrize("T", [1, 127, 300, 513])
@pytest.mark.parametrize("H,V", [(128, 256), (576, 640), (896, 9024), (192, 1000), (256, 20403), (72, 600)])
def test_against_float64(dev, T, H, V):
    g = torch.Generator().manual_seed(T + H + V)
    hidden = torch.randn(T, H, generator=g).bfloat16().to(dev)
    weight = (torch.randn(V, H, generator=g) * 0.1).bfloat16().to(dev)
    labels = torch.randint(0, V, (T,), generator=g).to(dev)
    labels[T // 2] = -100
    for temperature in (1.0, 0.7):
        got = compute_logprobs(hidden, weight, dict(rolled_input_ids=labels), temperature=temperature, pad_length=T // 3)
        want, tol = _want(hidden, weight, labels, temperature)
        n = T - T // 3
        assert got.shape == (n,) and (got.double() - want[:n]).abs().max().item() <= tol


def test_bias_through_the_adapter(dev):
    g = torch.Generator().manual_seed(3)
    lm = torch.nn.Module()
    lm.model = lambda hidden: hidden
    lm.lm_head = torch.nn.Linear(320, 1600, device=dev)
    hidden = torch.randn(200, 320, generator=g).bfloat16().to(dev)
    labels = torch.randint(0, 1600, (200,), generator=g).to(dev)
    adapter = FusedLMHeadAdapter(lm)
    adapter.module.model = lambda hidden, rolled_input_ids: hidden
    got = adapter.compute_logprobs(dict(hidden=hidden, rolled_input_ids=labels))
    want, tol = _want(hidden, lm.lm_head.weight.detach().bfloat16(), labels, bias=lm.lm_head.bias.detach())
    assert (got.double() - want).abs().max().item() <= tol


@pytest.mark.parametrize("V", [1536, 1600, 1000])
@pytest.mark.parametrize("rows", ["rising", "falling", "low", "hot"])
def test_rows_far_from_their_first_logits(dev, rows, V):
    T, H = 130, 128
    g = torch.Generator().manual_seed(V)
    hidden = torch.randn(T, H, generator=g).abs().bfloat16()
    v = torch.arange(V)
    scale = {"rising": v / V * 8, "falling": 8 - v / V * 8, "low": torch.full((V,), -6.0), "hot": torch.zeros(V)}[rows]
    weight = (torch.randn(V, H, generator=g) * 0.05).abs() * torch.sign(scale)[:, None] + scale[:, None] * 0.5
    if rows == "hot":
        weight = torch.randn(V, H, generator=g) * 0.05
        weight[V - 3] = 4.0
    weight, hidden = weight.bfloat16().to(dev), hidden.to(dev)
    labels = torch.randint(0, V, (T,), generator=g).to(dev)
    labels[::7] = V - 3
    want, tol = _want(hidden, weight, labels)
    got = compute_logprobs(hidden, weight, dict(rolled_input_ids=labels))
    assert (got.double() - want).abs().max().item() <= tol
    assert got.max().item() <= 0.0


def test_rows_that_are_not_finite_are_those_of_the_full_sweep(dev):
    T, H, V = 140, 128, 1536
    g = torch.Generator().manual_seed(0)
    hidden = torch.randn(T, H, generator=g).bfloat16().to(dev)
    weight = (torch.randn(V, H, generator=g) * 0.1).bfloat16().to(dev)
    hidden[3, 5], hidden[70, 0], hidden[139, 127] = float("nan"), float("inf"), float("-inf")
    labels = torch.randint(0, V, (T,), generator=g).to(dev)
    got = compute_logprobs(hidden, weight, dict(rolled_input_ids=labels))
    with torch.no_grad():
        full = fused_lm_head_logprobs_entropy(hidden, weight, labels).logprobs
    assert torch.equal(got.isnan(), full.isnan())
    ok = ~full.isnan()
    torch.testing.assert_close(got[ok], full[ok], rtol=1e-6, atol=1e-5)


@pytest.mark.parametrize("V", [40000, 151936])  # (several tiles of the vocabulary to a workgroup)
@pytest.mark.parametrize("lead", [12, 30, 40, 55])
def test_confident_tokens(dev, lead, V):
    """A label that stands alone, ``lead`` nats above normal logits. The logits are exact (one product each, of
    bf16 values), so the error is that of the sums: as near as the sweep with all outputs, and where nothing but the label
    counts (30 nats on) an ulp of its exponential and one of the sum, 2^-22."""
    T, H = 128, 128
    g = torch.Generator().manual_seed(lead + V)
    hidden, weight = torch.eye(T, H), torch.randn(V, H, generator=g)
    labels = torch.randint(0, V, (T,), generator=g)
    weight[labels, torch.arange(T)] = lead + torch.randn(T, generator=g)
    hidden, weight, labels = hidden.bfloat16().to(dev), weight.bfloat16().to(dev), labels.to(dev)
    want, _ = _want(hidden, weight, labels)
    got = compute_logprobs(hidden, weight, dict(rolled_input_ids=labels))
    with torch.no_grad():
        full = fused_lm_head_logprobs_entropy(hidden, weight, labels).logprobs
    error, of_full = ((x.double() - want).abs().max().item() for x in (got, full))
    assert error <= (2.0 ** -22 if lead >= 30 else 2.0 ** -22 + 1.5 * of_full), (error, of_full)
