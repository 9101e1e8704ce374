"""Advantages with a fixed lambda run as one launch in front of their normalisation; a lambda per row takes the
calls it was made of (reward scores, shaping, scan of padded rows). With the same lambda in both forms, the shaped
arrays are the same bits and what comes of the scan, whose row sums differ by the order in which the compiler adds
them, agrees to |difference| <= 64 * 2^-24 of the largest magnitude. (Both walk a row by the same code:
test_gpu_advantage_rows.py has the scan against the oracle.)

Row lengths around a thread's 8 tokens and the tile, none a multiple of anything; rows without tokens, with one,
with two, full ones; arrays at any address; every estimator; scores shaped, normalised in groups (whole, ragged, one
row) or given."""

import pytest
import torch

from areal_amd.config import NormConfig
from areal_amd.data import KLEstimator, Normalization
from areal_amd.ppo.actor import compute_advantages

pytestmark = pytest.mark.gpu


def _odd(x, shift):
    """The same values in a contiguous tensor that starts `shift` elements into an allocation."""
    flat = torch.empty(x.numel() + shift, dtype=x.dtype, device=x.device)
    flat[shift:] = x.reshape(-1)
    return flat[shift:].view(x.shape)


def _batch(dev, bs, L, ref, critic, shift):
    g = torch.Generator().manual_seed(1000 * bs + L)
    lens = torch.randint(0, L + 1, (bs,), generator=g)
    lens[0], lens[-1] = L, 0
    if bs > 4:
        lens[1], lens[2] = min(1, L), min(2, L)
    pos = torch.arange(L)[None]
    attn = pos < lens[:, None]
    normal = lambda: torch.randn(bs, L, generator=g)  # noqa: E731
    data = dict(input_ids=torch.zeros(bs, L, dtype=torch.long), attention_mask=attn,
                loss_mask=attn & (torch.rand(bs, L, generator=g) > 0.3), logprobs=normal() - 1, prox_logp=normal() - 1,
                rewards=torch.randn(bs, generator=g) * 3)
    if ref:
        data["ref_logp"] = normal() - 1
    if critic:
        data["values"] = normal()
    return {k: _odd(v.to(dev), shift) for k, v in data.items()}


@pytest.mark.parametrize("bs,L", [(1, 1), (5, 2), (8, 7), (8, 8), (16, 9), (6, 200), (9, 1001), (4, 2047), (8, 2048), (8, 2049),
                                  (3, 2057), (5, 8195), (1030, 1793)])
@pytest.mark.parametrize("variant", range(6))
def test_same_as_the_separate_calls(dev, bs, L, variant):
    ref, critic, shift = variant % 2 == 0, variant in (0, 3, 5), (0, 1, 3)[variant % 3]
    norms = [NormConfig(mean_level="group", std_level="group", group_size=4),
             NormConfig(mean_level="group", std_level=None, group_size=1),
             NormConfig(mean_level="batch", std_level="batch", group_size=1)]
    options = dict(
        kl_ctl=0.1, kl_estimator=KLEstimator(("k1", "k2", "k3")[variant % 3], apply_clamp=variant != 4), discount=0.97,
        reward_bias=0.1, reward_scaling=1.5, reward_clip=2.0, mask_no_eos_with_zero=variant == 1,
        reward_norm=Normalization(norms[variant % 3]) if variant != 4 else None, adv_norm=Normalization(norms[0]),
        recompute_logprob=variant in (2, 5), use_decoupled_loss=variant == 3,
        group_sizes=[bs - 1, 1] if variant == 5 and bs > 1 else None)
    one, many = _batch(dev, bs, L, ref, critic, shift), _batch(dev, bs, L, ref, critic, shift)
    compute_advantages(one, gae_lambda=0.9, **options)
    compute_advantages(many, gae_lambda=torch.full((bs,), 0.9, device=dev), **options)
    for k in ("loss_mask", "logprobs", "kl_rewards", "tot_rewards", "prox_logp", "ref_logp"):
        if k in many:
            assert torch.equal(one[k], many[k]), k
    for k in ("returns", "advantages"):
        assert (one[k] - many[k]).abs().max().item() <= 2.0 ** -18 * (1 + many[k].abs().max().item()), k
