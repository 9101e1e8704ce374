"""No call has a forward-mode formula: an input with a tangent is refused, also where no gradient is asked for and
the call makes no autograd node. Needs no GPU: tangents are looked for first."""

import pytest
import torch
import torch.autograd.forward_ad as fwad

from areal_amd.functional import cispo_loss_fn, fused_lm_head_logprobs_entropy, ppo_actor_loss_fn, ppo_critic_loss_fn
from areal_amd.functional.aux_losses import sapo_loss_fn

Z, MASK = torch.zeros(6), torch.ones(6, dtype=torch.bool)
LOSSES = dict(
    ppo=lambda x: ppo_actor_loss_fn(x, Z, None, Z, 0.2, MASK),
    cispo=lambda x: cispo_loss_fn(x, Z, Z, 1.0, MASK, eps_clip_higher=0.2),
    sapo=lambda x: sapo_loss_fn(x, Z, Z, 1.0, 1.05, MASK),
    critic=lambda x: ppo_critic_loss_fn(x, Z, Z, 0.2, MASK),
)


@pytest.mark.parametrize("loss", LOSSES)
def test_losses(loss):
    with fwad.dual_level(), pytest.raises(NotImplementedError):
        LOSSES[loss](fwad.make_dual(torch.zeros(6), torch.ones(6)))


@pytest.mark.parametrize("dual", ["hidden", "weight", "bias"])
def test_lm_head_without_gradients(dual):
    x = dict(hidden=torch.zeros(6, 8).bfloat16(), weight=torch.zeros(10, 8).bfloat16(), bias=torch.zeros(10))
    with fwad.dual_level(), torch.no_grad(), pytest.raises(NotImplementedError):
        x[dual] = fwad.make_dual(x[dual], torch.ones_like(x[dual]))
        fused_lm_head_logprobs_entropy(x["hidden"], x["weight"], torch.zeros(6, dtype=torch.long), bias=x["bias"])
