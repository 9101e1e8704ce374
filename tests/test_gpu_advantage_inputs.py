"""Inputs of the advantage calls off the common path: the no-EOS mask of turn-level GAE in host memory."""

import pytest
import torch

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
