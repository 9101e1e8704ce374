"""The row scan's quads (4 tokens a thread, 256 a wave, a second quad 256 tokens on, 512 a wave, 2048 a tile) and both
sides of the rule on the number of rows: one-launch advantages against the
separate calls, which a lambda per row takes. The shaped arrays are the same bits, the scan differs by fp32 rounding:
20 compositions of maps, |difference| <= 64 * 2^-24 of the largest magnitude."""

import pytest
import torch

from areal_amd.config import NormConfig
from areal_amd.data import KLEstimator, Normalization
from areal_amd.ppo.actor import compute_advantages

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs,L", [(1024, 3), (1025, 1791), (1025, 1792), (4, 4), (4, 5), (4, 255), (4, 256), (4, 257), (4, 260), (4, 511), (4, 513), (4, 2044), (4, 2053),
                                  (4, 4096), (4, 4099)])
def test_rows_and_quads(dev, bs, L):
    g = torch.Generator().manual_seed(bs + L)
    lens = torch.randint(1, L + 1, (bs,), generator=g)
    lens[0] = L
    attn = torch.arange(L)[None] < lens[:, None]
    data = dict(input_ids=torch.zeros(bs, L, dtype=torch.long), attention_mask=attn,
                loss_mask=attn & (torch.rand(bs, L, generator=g) > 0.3), logprobs=torch.randn(bs, L, generator=g) - 1,
                ref_logp=torch.randn(bs, L, generator=g) - 1, values=torch.randn(bs, L, generator=g),
                rewards=torch.randn(bs, generator=g))
    options = dict(kl_ctl=0.1, kl_estimator=KLEstimator("k1"), discount=0.97,
                   adv_norm=Normalization(NormConfig(mean_level="group", std_level="group", group_size=1)))
    one = {k: v.to(dev) for k, v in data.items()}
    many = {k: v.to(dev) for k, v in data.items()}
    compute_advantages(one, gae_lambda=0.9, **options)
    compute_advantages(many, gae_lambda=torch.full((bs,), 0.9, device=dev), **options)
    for k in ("loss_mask", "logprobs", "kl_rewards", "tot_rewards", "ref_logp"):
        assert torch.equal(one[k], many[k]), k
    assert (one["returns"] - many["returns"]).abs().max().item() <= 2.0 ** -18 * many["returns"].abs().max().item()
    # rows of one or two active tokens have a deviation near eps: an ulp of the mean there is of order one
    full = one["loss_mask"].sum(1) > 8
    diff = (one["advantages"] - many["advantages"])[full]
    assert diff.numel() == 0 or diff.abs().max().item() <= 2.0 ** -16 * many["advantages"][full].abs().max().item()
