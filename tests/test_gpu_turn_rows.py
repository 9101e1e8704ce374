"""Turn-level GAE at the edges of its blocks (1024, 2048 and 4096 tokens a tile, 4 a thread) and of the turns a row keeps
in LDS (512), against the oracle (fp32 recurrence, fp64 prefix sums: 1e-5)."""

import pytest
import torch

from areal_amd.config import NormConfig
from areal_amd.data import KLEstimator, Normalization
from areal_amd.ppo.actor import compute_advantages
from oracle import gae as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("critic", [False, True])
@pytest.mark.parametrize("bs,L,turn", [(4, 1, 1), (4, 3, 1), (4, 4, 2), (4, 5, 2), (4, 1023, 100), (4, 1024, 7), (4, 1025, 300),
                                       (4, 2047, 4), (4, 2049, 4), (4, 2052, 4), (4, 4096, 8), (4, 4097, 8), (4, 4100, 7),
                                       (4, 9001, 300), (4, 700, 1), (4, 5000, 3),
                                       (1024, 1025, 300), (1028, 1025, 300), (512, 2049, 7), (516, 2049, 7)])
def test_rows_of_one_tile_and_more(dev, bs, L, turn, critic):
    g = torch.Generator().manual_seed(L + turn)
    lens = torch.tensor([L, max(1, L - 1), max(1, L // 2), 1]).repeat(bs // 4)
    pos = torch.arange(L)[None]
    attn = pos < lens[:, None]
    data = dict(input_ids=torch.zeros(bs, L, dtype=torch.long), attention_mask=attn,
                loss_mask=attn & (torch.rand(bs, L, generator=g) > 0.2) & (pos > 0), logprobs=torch.randn(bs, L, generator=g),
                rewards=torch.randn(bs, generator=g),
                turn_ids=torch.where(attn, (pos // turn).expand(bs, L), -1).to(torch.int32))
    if critic:
        data["values"] = torch.randn(bs, L, generator=g)
    out = compute_advantages({k: v.to(dev) for k, v in data.items()}, kl_ctl=0.0, kl_estimator=KLEstimator("k1"),
                             adv_norm=Normalization(NormConfig(mean_level=None, std_level=None, group_size=1)),
                             discount=0.9, gae_lambda=0.8, gae_timestep_unit="turn")
    mask = out["loss_mask"].cpu().float()
    ids = torch.cat([data["turn_ids"][:, 1:], torch.full((bs, 1), -1, dtype=torch.int32)], 1)
    rewards = out["tot_rewards"].cpu()
    values = data.get("values", torch.zeros(bs, L))
    want_adv, want_ret = G.gae_turn_level(rewards, values, mask, ids, lens == L, 0.9, 0.8)
    torch.testing.assert_close(out["advantages"].cpu(), want_adv, rtol=1e-5, atol=1e-5 * max(1.0, want_adv.abs().max().item()))
    torch.testing.assert_close(out["returns"].cpu(), want_ret, rtol=1e-5, atol=1e-5 * max(1.0, want_ret.abs().max().item()))
