"""A loss kernel reads as many elements of each array as the loss mask (the critic's value) has, reward shaping as
many as the batch has rows and slots: an array of another size is refused before any kernel could read past its end.
Needs no GPU: sizes are compared first."""

import pytest
import torch

from areal_amd import _lib
from areal_amd.functional import cispo_loss_fn, ppo_actor_loss_fn, ppo_critic_loss_fn
from areal_amd.functional.aux_losses import sapo_loss_fn
from areal_amd.ppo.actor import compute_advantages, grpo_loss_fn

N = 6
MASK = torch.ones(N, dtype=torch.bool)
SIZES = [1, N - 1, N + 1]


def _arrays(name, size, *names):
    return [torch.zeros(size if n == name else N) for n in names]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("name", ["logprobs", "proximal_logprobs", "advantages"])
def test_actor_losses(name, size):
    lp, prox, adv = _arrays(name, size, "logprobs", "proximal_logprobs", "advantages")
    match = f"{name} has {size} elements, expected {N}"
    with pytest.raises(_lib.ArealHipError, match=match):
        ppo_actor_loss_fn(lp, prox, None, adv, 0.2, MASK)
    with pytest.raises(_lib.ArealHipError, match=match):
        cispo_loss_fn(lp, prox, adv, 1.0, MASK, eps_clip_higher=0.2)


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("stats_mode", ["tensors", "reduced"])
def test_logged_old_logprobs(stats_mode, size):
    z = torch.zeros(N)
    data = dict(logprobs=torch.zeros(size), prox_logp=z, advantages=z, loss_mask=MASK)
    with pytest.raises(_lib.ArealHipError, match=f"old_logprobs has {size} elements, expected {N}"):
        grpo_loss_fn(z, z, data, eps_clip=0.2, eps_clip_higher=None, c_clip=None, stats={}, stats_mode=stats_mode)


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("name", ["logprobs", "old_logprobs", "advantages"])
def test_sapo_loss(name, size):
    lp, old, adv = _arrays(name, size, "logprobs", "old_logprobs", "advantages")
    with pytest.raises(_lib.ArealHipError, match=f"{name} has {size} elements, expected {N}"):
        sapo_loss_fn(lp, old, adv, 1.0, 1.05, MASK)


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("name", ["old_value", "target_value", "loss_mask"])
def test_critic_loss(name, size):
    value, old, target, mask = _arrays(name, size, "value", "old_value", "target_value", "loss_mask")
    with pytest.raises(_lib.ArealHipError, match=f"{name} has {size} elements, expected {N}"):
        ppo_critic_loss_fn(value, old, target, 0.2, mask)


@pytest.mark.parametrize("rows", [1, 2, 4])
@pytest.mark.parametrize("name", ["rewards", "logprobs", "loss_mask", "attention_mask", "ref_logp"])
def test_advantages(name, rows):
    bs, length = 3, 5
    z = torch.zeros(bs, length)
    data = dict(input_ids=z.long(), rewards=torch.zeros(bs), logprobs=z, loss_mask=z > 0, attention_mask=z > 0, ref_logp=z)
    data[name] = data[name][:1].expand(rows, *data[name].shape[1:]).contiguous()
    n = data[name].numel()
    with pytest.raises(_lib.ArealHipError, match=f"{name} has {n} elements, expected {bs if name == 'rewards' else bs * length}"):
        compute_advantages(data)
