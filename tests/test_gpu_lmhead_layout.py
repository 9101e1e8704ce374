"""Layout of the lm_head launches over the XCDs at the token counts where it changes: one B tile
and several, whole and ragged ones (a wave without tokens, a wave with one), more copies of dHidden's
vocabulary range than XCDs, and a vocabulary whose last tile overlaps its predecessor.

The bound on the gradients is bf16's: dlogits are rounded to bf16 (2^-9 relative) before they are
contracted and the result once more, so the 2-norm error is below 2 * 2^-8. The log-probabilities are
fp32 sums of products of bf16 values."""

import pytest
import torch

from areal_amd.functional import fused_lm_head_logprobs_entropy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("save_probs", [True, False])
@pytest.mark.parametrize("tokens", [1, 127, 128, 129, 256, 257, 384, 509, 900, 2049])
@pytest.mark.parametrize("hidden_size,vocab", [(128, 9024), (896, 6400), (576, 640)])
def test_ragged_token_counts_match_fp32(tokens, hidden_size, vocab, save_probs):
    dev = torch.device("cuda", 0)
    g = torch.Generator().manual_seed(tokens)
    hidden = torch.randn(tokens, hidden_size, generator=g).bfloat16().to(dev).requires_grad_(True)
    weight = (torch.randn(vocab, hidden_size, generator=g) * 0.1).bfloat16().to(dev).requires_grad_(True)
    labels = torch.randint(0, vocab, (tokens,), generator=g).to(dev)
    grad = torch.randn(tokens, generator=g).to(dev)
    out = fused_lm_head_logprobs_entropy(hidden, weight, labels, save_probs=save_probs)
    out.logprobs.backward(grad)

    h32 = hidden.detach().float().requires_grad_(True)
    w32 = weight.detach().float().requires_grad_(True)
    logp = torch.log_softmax(h32 @ w32.t(), -1)
    want = logp.gather(1, labels[:, None])[:, 0]
    want.backward(grad)
    entropy = -(logp.exp() * logp).sum(-1)
    assert torch.allclose(out.logprobs, want, atol=1e-4, rtol=1e-5)
    assert torch.allclose(out.entropy, entropy, atol=1e-4, rtol=1e-5)
    for got, ref in ((hidden.grad, h32.grad), (weight.grad, w32.grad)):
        assert (got.float() - ref).norm() <= 2.0 ** -7 * ref.norm()
