"""The loss stage where its layout changes: sequences around the number and length from which a wave
takes one, alignments that rule out 16-byte loads, batches around one wave and around the four-token form,
and what the loss kernel does besides the loss (fp32 copies of the masks, statistics of the proximal
log-probs, tokens that are not finite)."""

import pytest
import torch

from areal_amd.config import RejectionSamplingConfig
from areal_amd.functional import apply_rejection_sampling
from areal_amd.ppo.actor import grpo_loss_fn
from areal_amd.stats import masked_stats
from oracle.loss import rejection_sampling

pytestmark = pytest.mark.gpu


def _batch(lens, offset, seed=0):
    """Arrays that start ``offset`` elements behind an aligned address."""
    dev = torch.device("cuda", 0)
    n = sum(lens)
    g = torch.Generator().manual_seed(seed)

    def moved(x):
        buf = torch.zeros(n + offset, dtype=x.dtype, device=dev)
        buf[offset:] = x.to(dev)
        return buf[offset:]

    prox = moved(torch.randn(n, generator=g) * 0.5 - 1)
    old = moved(prox.cpu() + 0.1 * torch.randn(n, generator=g))
    mask = moved(torch.rand(n, generator=g) > 0.3)
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device=dev)
    return prox, old, mask, cu, g


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("lens", [[1], [3, 0, 5], [64, 1, 63, 200], [1023, 1025, 4096, 2], [4097, 900, 5000], [7] * 700])
@pytest.mark.parametrize("metric,agg", [("kl_k2", "mean"), ("kl_k3", "max"), ("ratio", "mean"), ("kl_k1", "sum")])
def test_sequence_rejection(lens, offset, metric, agg):
    prox, old, mask, cu, _ = _batch(lens, offset)
    # a bound between the per-sequence values: those of random sequences are not within rounding of it
    upper = {"kl_k2": 0.0051, "kl_k3": 0.021, "ratio": 1.003, "kl_k1": 0.37}[metric]
    cfg = RejectionSamplingConfig(level="sequence", action="mask", metric=metric, agg=agg, upper=upper)
    got = apply_rejection_sampling(prox, old, mask, cu, cfg)
    lengths = [n for n in lens if n > 0]  # the oracle indexes sequences by their first token
    cu_ref = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32)
    want = rejection_sampling(prox.cpu(), old.cpu(), mask.cpu(), cu_ref, level="sequence", metric=metric, agg=agg,
                              upper=upper)
    assert torch.equal(got.loss_mask.cpu(), want.loss_mask)
    torch.testing.assert_close(got.behave_imp_weight.cpu(), want.behave_imp_weight, rtol=1e-5, atol=1e-6)


# 16 waves a sequence up to 512 of at least 512 tokens on average, 8 up to 2048, 4 beyond; a step of a block is 4096, 2048, 1024 tokens
@pytest.mark.parametrize("lens", [[4095, 4096, 4097, 0, 1], [511, 512] * 100 + [20000], [512] * 512, [513] * 513, [2047, 0, 2049] * 300,
                                  [512] * 2048, [515] * 2049])
@pytest.mark.parametrize("metric,agg", [("kl_k2", "mean"), ("kl_k3", "max"), ("ratio", "mean")])
def test_sequence_rejection_of_long_sequences(lens, metric, agg):
    test_sequence_rejection(lens, 0, metric, agg)


# more than 4096 sequences take a wave each up to a mean of 384 tokens
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("lens", [[7] * 4096, [7, 1, 0, 300] * 1025, [2, 5000] + [65] * 4095, [384] * 4097, [385] * 4097])
@pytest.mark.parametrize("metric,agg", [("kl_k2", "mean"), ("ratio", "mean")])
def test_sequence_rejection_of_many_sequences(lens, offset, metric, agg):
    test_sequence_rejection(lens, offset, metric, agg)


# such a wave reads four steps of 256 tokens (64 unaligned) at once while its lanes have them
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("metric,agg", [("kl_k2", "mean"), ("kl_k3", "max")])
def test_sequence_rejection_of_waves_with_several_steps(offset, metric, agg):
    lens = [255, 257, 1023, 1024, 1025, 1027, 1028, 769, 2047, 2049, 5, 4100] + [3, 2] * 2050
    test_sequence_rejection(lens, offset, metric, agg)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("n", [1, 63, 65, 4097, 262144, 262147])
@pytest.mark.parametrize("cispo", [False, True])
@pytest.mark.parametrize("rejection", [False, True])
def test_logged_tensors_and_reduced_statistics_agree(n, offset, cispo, rejection):
    prox, old, mask, cu, g = _batch([n], offset)
    dev = prox.device
    lp = (prox + 0.1 * torch.randn(n, generator=g).to(dev)).requires_grad_(True)
    data = dict(logprobs=old, prox_logp=prox, advantages=torch.randn(n, generator=g).to(dev), loss_mask=mask,
                cu_seqlens=cu)
    rs = RejectionSamplingConfig(level="token", action="mask", metric="ratio", lower=0.8, upper=1.2)
    kw = dict(eps_clip=0.2, eps_clip_higher=0.28, c_clip=None, rejection_sampling=rs if rejection else None,
              use_cispo_loss=cispo)
    entropy = torch.rand(n, generator=g).to(dev)
    tensors, reduced = {}, {}
    loss = grpo_loss_fn(lp, entropy, data, stats=tensors, **kw)
    loss_r = grpo_loss_fn(lp, entropy, data, stats=reduced, stats_mode="reduced", **kw)
    bare = grpo_loss_fn(lp, entropy, data, **kw)
    assert torch.equal(loss, loss_r) and torch.equal(loss, bare)
    diff = (old - lp.detach()) * mask
    assert torch.equal(tensors["logp_diff"], diff) and torch.equal(tensors["logp_abs_diff"], diff.abs())
    assert torch.equal(tensors["clip_ratio"], tensors["clipped_tokens"].float())
    assert torch.equal(tensors["dual_clip_ratio"], tensors["dual_clipped_tokens"].float())
    den = mask
    if rejection:
        den = tensors["unclipped_behave_tokens"]
        assert torch.equal(tensors["behave_filtered_ratio"], (mask & ~den).float())
    got = reduced["compute_logp/prox_logp_gt"]
    want = masked_stats({"x": prox}, {"x": den})["x"]
    assert got["count"] == want["count"] == reduced["denominator/compute_logp/n_valid_tokens"]
    if got["count"] > 0:
        # fp32 sums of at most 16 x 16 tokens, fp64 from there
        assert abs(got["sum"] - want["sum"]) <= 256 * 2.0 ** -24 * prox.abs().sum().item()
        assert (got["min"], got["max"]) == (want["min"], want["max"])


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("sapo", [False, True])
def test_proximal_log_prob_that_is_not_finite(value, sapo):
    prox, old, mask, cu, g = _batch([3000], 0)
    lp = prox.clone().requires_grad_(True)
    prox[2999], mask[2999] = value, False  # outside the loss mask: it counts all the same
    data = dict(logprobs=old, prox_logp=prox, advantages=torch.ones_like(old), loss_mask=mask, cu_seqlens=cu)
    kw = dict(eps_clip=0.2, eps_clip_higher=None, c_clip=None, use_sapo_loss=sapo)
    with pytest.raises(RuntimeError, match="prox_logp contains NaN or Inf"):
        grpo_loss_fn(lp, torch.zeros_like(lp), data, **kw)
    if not sapo:
        assert torch.isnan(grpo_loss_fn(lp, torch.zeros_like(lp), data, defer_host_reads=True, **kw))


@pytest.mark.parametrize("lens", [[1], [3, 0, 5], [1, 2, 3, 4, 5, 6, 7, 8, 9] * 30, [2, 0, 0, 1, 3] * 60000, [262144, 1, 5]])
@pytest.mark.parametrize("level", ["token", "sequence"])
@pytest.mark.parametrize("offset", [0, 1])
def test_gradient_does_not_depend_on_what_is_logged(lens, level, offset):
    """Several sequences inside a thread's four tokens, empty ones among them; bit for bit."""
    prox, old, mask, cu, g = _batch(lens, offset)
    n, dev = prox.numel(), prox.device
    lp = (prox + 0.1 * torch.randn(n, generator=g).to(dev)).requires_grad_(True)
    data = dict(logprobs=old, prox_logp=prox, advantages=torch.randn(n, generator=g).to(dev), loss_mask=mask,
                cu_seqlens=cu)
    rs = (RejectionSamplingConfig(level="token", action="mask", metric="ratio", lower=0.9, upper=1.1) if level == "token"
          else RejectionSamplingConfig(level="sequence", action="clamp", metric="ratio", agg="mean", upper=1.003))
    results = []
    for stats, mode in ((None, "tensors"), ({}, "tensors"), ({}, "reduced")):
        lp.grad = None
        loss = grpo_loss_fn(lp, torch.zeros(n, device=dev), data, eps_clip=0.2, eps_clip_higher=None, c_clip=None,
                            rejection_sampling=rs, stats=stats, stats_mode=mode)
        loss.backward()
        results.append((loss.detach(), lp.grad))
    for loss, grad in results[1:]:
        assert torch.equal(grad, results[0][1])
        torch.testing.assert_close(loss, results[0][0], rtol=1e-6, atol=1e-7)  # (other blocks: fp64 sums in another order)
