"""Normalised reward scores either side of the row count up to which the one launch of the advantages makes them itself
(2048 rows): one group of nearly all rows, whole groups with a ragged last one, and a normalisation without levels (one
group of all rows), against the oracle."""

import pytest
import torch

from areal_amd import _lib
from areal_amd.config import NormConfig
from areal_amd.data import KLEstimator, Normalization
from areal_amd.ppo.actor import compute_advantages
from oracle import norm as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", ["long", "ragged", "none"])
@pytest.mark.parametrize("bs", [1537, 2047, 2048, 2049])
def test_scores_of_many_rows(dev, monkeypatch, bs, groups):
    L = 1793
    g = torch.Generator().manual_seed(bs)
    attn = torch.ones(bs, L, dtype=torch.bool)
    rewards = torch.randn(bs, generator=g)
    data = dict(input_ids=torch.zeros(bs, L, dtype=torch.long), attention_mask=attn, loss_mask=attn,
                logprobs=torch.randn(bs, L, generator=g), rewards=rewards)
    level = None if groups == "none" else "group"
    config = dict(mean_level=level, std_level=level, group_size=16)
    sizes = [bs - 3, 3] if groups == "long" else None
    host, one_launch = _lib.host(), []
    prep = host.advantage_prep

    def spy(*args):
        res = prep(*args)
        one_launch.append(res[-1] is not None)
        return res

    monkeypatch.setattr(host, "advantage_prep", spy)
    out = compute_advantages({k: v.to(dev) for k, v in data.items()}, kl_ctl=0.0, kl_estimator=KLEstimator("k1"),
                             reward_norm=Normalization(NormConfig(**config)), reward_bias=0.1, reward_scaling=1.5,
                             reward_clip=2.0, discount=0.97, gae_lambda=0.9, group_sizes=sizes,
                             adv_norm=Normalization(NormConfig(mean_level=None, std_level=None, group_size=1)))
    assert one_launch == [True]
    shaped = ((rewards + 0.1) * 1.5).clip(-2.0, 2.0)
    want = N.normalization(shaped, **config, group_sizes=sizes)
    torch.testing.assert_close(out["tot_rewards"][:, L - 2].cpu(), want, rtol=1e-5, atol=1e-5)
    assert out["tot_rewards"].count_nonzero().item() == want.count_nonzero().item()
