"""The row scan's quads (4 tokens a thread, 256 a wave, a second quad 256 tokens on, 512 a wave, 2048 a tile) and both
sides of the rule on the number of rows. One-launch advantages against the separate calls, which a lambda per row takes:
the shaped arrays are the same bits; the scan of rows that both walk is the same code, its sums ride in another
launch. And against the oracle: the scan itself, whichever launch it is in."""


import pytest
import torch

from areal_amd import _lib
from areal_amd.config import NormConfig
from areal_amd.data import KLEstimator, Normalization
from areal_amd.ppo.actor import compute_advantages
from oracle import gae as G

pytestmark = pytest.mark.gpu


SHAPES = [(1024, 3), (1025, 1791), (1025, 1792), (4, 4), (4, 5), (4, 255), (4, 256), (4, 257), (4, 260), (4, 511), (4, 513),
          (4, 2044), (4, 2053), (4, 4096), (4, 4099)]


@pytest.mark.parametrize("bs,L", SHAPES)
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


@pytest.mark.parametrize("lam", ["number", "per row"])
@pytest.mark.parametrize("critic", [False, True])
@pytest.mark.parametrize("bs,L", SHAPES + [(1, 1), (5, 2), (8, 7), (6, 200), (9, 1001), (4, 2047), (8, 2048), (8, 2049), (5, 8195)])
def test_scan_against_the_oracle(dev, monkeypatch, bs, L, critic, lam):
    """Returns and advantages (nothing normalised) of an fp32 recurrence: 1e-5 of the largest magnitude. A number for lambda
    goes through the one launch exactly where the rule says so."""
    g = torch.Generator().manual_seed(3 * bs + L)
    lens = torch.randint(0, L + 1, (bs,), generator=g)
    lens[0], lens[-1] = L, 1
    attn = torch.arange(L)[None] < lens[:, None]
    data = dict(input_ids=torch.zeros(bs, L, dtype=torch.long), attention_mask=attn,
                loss_mask=attn & (torch.rand(bs, L, generator=g) > 0.3), logprobs=torch.randn(bs, L, generator=g) - 1,
                ref_logp=torch.randn(bs, L, generator=g) - 1, rewards=torch.randn(bs, generator=g))
    if critic:
        data["values"] = torch.randn(bs, L, generator=g)
    values = data.get("values", torch.zeros(bs, L))
    host, one_launch = _lib.host(), []
    prep = host.advantage_prep

    def spy(*args):
        res = prep(*args)
        one_launch.append(res[-1] is not None)
        return res

    monkeypatch.setattr(host, "advantage_prep", spy)
    out = compute_advantages({k: v.to(dev) for k, v in data.items()}, kl_ctl=0.1, kl_estimator=KLEstimator("k1"),
                             discount=0.97, gae_lambda=0.9 if lam == "number" else torch.full((bs,), 0.9, device=dev),
                             adv_norm=Normalization(NormConfig(mean_level=None, std_level=None, group_size=1)))
    assert one_launch == [lam == "number" and (L >= 1792 or bs <= 1024)]
    mask = torch.roll(data["loss_mask"], -1, 1).float()
    assert torch.equal(out["loss_mask"].cpu(), mask)
    want_adv, want_ret = G.gae_padded(out["tot_rewards"].cpu(), values, mask, lens == L, 0.97, 0.9)
    # (a normalisation without levels still leaves the masked tokens out)
    for got, want in ((out["advantages"], want_adv * mask), (out["returns"], want_ret)):
        assert (got.cpu() - want).abs().max().item() <= 1e-5 * max(1.0, want.abs().max().item())
