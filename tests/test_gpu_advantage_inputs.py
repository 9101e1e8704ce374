"""Inputs of the advantage calls off the common path: the no-EOS mask of turn-level GAE in host memory, arrays
that are refused there, log-probabilities that are not finite, a negative reward clip, more reward scores than 2^24."""

import pytest
import torch

from areal_amd import _lib
from areal_amd.config import NormConfig
from areal_amd.data import KLEstimator, Normalization
from areal_amd.ppo.actor import compute_advantages
from areal_amd.ppo.gae import _compute_turn_level_gae

pytestmark = pytest.mark.gpu


def test_turn_gae_moves_its_no_eos_mask(dev):
    g = torch.Generator().manual_seed(1)
    bs, length = 5, 300
    ids = (torch.arange(length) // 50).to(torch.int32).expand(bs, length).contiguous()
    no_eos = torch.tensor([True, False, True, False, True])
    x = [t.to(dev) for t in (torch.randn(bs, length, generator=g), torch.randn(bs, length, generator=g),
                             (torch.rand(bs, length, generator=g) > 0.2).float(), ids)]
    want = _compute_turn_level_gae(*x, no_eos.to(dev), 0.99, 0.9)
    got = _compute_turn_level_gae(*x, no_eos, 0.99, 0.9)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("n,clip,group", [(37, -0.5, 0), (37, -0.5, 4), (2**24 + 3, 1.5, 0), (2**24 + 3, 1.5, 16)])
def test_reward_scores(dev, n, clip, group):
    """Bitwise the tensor operations when nothing is normalised; a group's scores against fp64."""
    x = torch.randn(n, device=dev, generator=torch.Generator(dev).manual_seed(n))
    x[5] = float("nan")
    groups = n // group if group else 0
    offsets = torch.arange(groups + 1, device=dev, dtype=torch.int64) * group
    rows = torch.full((groups,), group, device=dev, dtype=torch.int64)
    out = torch.empty_like(x)
    rc = _lib.load().areal_reward_scores(
        _lib.ptr(x), n, 0.25, 2.0, clip, _lib.ptr(offsets) if groups else None, _lib.ptr(rows) if groups else None,
        groups, -1, 2, 2, 1, 1e-5, _lib.ptr(out), _lib.stream_ptr(x.device))
    _lib.check(rc, "areal_reward_scores")
    want = torch.clip((x + 0.25) * 2.0, min=-clip, max=clip)
    if groups:
        w = want[: groups * group].double().view(groups, group)
        want[: groups * group] = ((w - w.mean(1, keepdim=True)) / (w.std(1, keepdim=True) + 1e-5)).float().view(-1)
        torch.testing.assert_close(out, want, rtol=1e-5, atol=1e-5, equal_nan=True)
    else:
        assert torch.equal(out.nan_to_num(7.0), want.nan_to_num(7.0))


def _batch(dev, bs, length):
    g = torch.Generator().manual_seed(bs)
    attn = torch.ones(bs, length, dtype=torch.bool)
    data = dict(input_ids=torch.zeros(bs, length, dtype=torch.long), attention_mask=attn, loss_mask=attn,
                logprobs=torch.randn(bs, length, generator=g), ref_logp=torch.randn(bs, length, generator=g),
                values=torch.randn(bs, length, generator=g), rewards=torch.randn(bs, generator=g),
                turn_ids=(torch.arange(length) // 10).to(torch.int32).expand(bs, length).contiguous())
    return {k: v.to(dev) for k, v in data.items()}


@pytest.mark.parametrize("unit", ["token", "turn"])
@pytest.mark.parametrize("name", ["ref_logp", "values", "logprobs", "loss_mask", "attention_mask", "rewards"])
def test_arrays_in_host_memory_are_refused(dev, name, unit):
    data = _batch(dev, 6, 100)
    data[name] = data[name].cpu()
    with pytest.raises(_lib.ArealHipError, match="MI355X only"):
        compute_advantages(data, kl_ctl=0.1, kl_estimator=KLEstimator("k1"), gae_timestep_unit=unit,
                           adv_norm=Normalization(NormConfig(mean_level="group", std_level="group", group_size=2)))


def test_token_ids_in_host_memory(dev):
    """Nothing reads them: the groups' tables go where the rewards are."""
    options = dict(kl_ctl=0.1, kl_estimator=KLEstimator("k1"))
    here, there = _batch(dev, 6, 100), _batch(dev, 6, 100)
    there["input_ids"] = there["input_ids"].cpu()
    for data in (here, there):
        norm = Normalization(NormConfig(mean_level="group", std_level="group", group_size=3))
        compute_advantages(data, reward_norm=norm, adv_norm=norm, **options)
    assert torch.equal(here["advantages"], there["advantages"])


@pytest.mark.parametrize("unit", ["token", "turn"])
@pytest.mark.parametrize("estimator", ["k1", "k2", "k3"])
@pytest.mark.parametrize("length", [100, 2051])
def test_logprobs_that_are_not_finite(dev, length, estimator, unit):
    """The clamped estimate keeps NaN, as ``torch.clamp`` does, and bounds the infinities."""
    data = _batch(dev, 6, length)
    data["loss_mask"][:, 0] = False  # (a prompt: no turn)
    data["logprobs"][0, 7], data["logprobs"][1, 50], data["ref_logp"][2, length - 3] = float("nan"), float("-inf"), float("nan")
    data["logprobs"][3, 20], data["ref_logp"][4, 30] = 30.0, float("-inf")
    estimate = KLEstimator(estimator)
    out = compute_advantages(data, kl_ctl=0.1, kl_estimator=estimate, gae_timestep_unit=unit,
                             adv_norm=Normalization(NormConfig(mean_level="group", std_level="group", group_size=2)))
    want = -0.1 * estimate(out["logprobs"], out["ref_logp"])
    assert want.isnan().any() and want.abs().eq(1.0).any()
    torch.testing.assert_close(out["kl_rewards"], want, rtol=1e-6, atol=1e-7, equal_nan=True)
