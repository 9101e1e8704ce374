"""The advantage kernels where their layout changes: rows around a 2048-token tile, groups that share a
4096-element block of the packed normalisation or end exactly at one, a batch without values, and the
one-launch reward scores; against the oracle (fp32 recurrences, fp64 sums: 1e-5 of the largest value)."""

import pytest
import torch

from areal_amd import _lib
from areal_amd.config import NormConfig
from areal_amd.data import KLEstimator, Normalization
from areal_amd.ppo import actor
from areal_amd.ppo.actor import compute_advantages
from areal_amd.ppo.gae import compute_gae_packed_normalized
from oracle import gae as G
from oracle import norm as N

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _close(got, want):
    torch.testing.assert_close(got.cpu(), want, rtol=1e-5, atol=1e-5 * max(1.0, want.abs().max().item()))


@pytest.mark.parametrize("levels", [("group", "group"), ("batch", "batch"), ("batch", "group"), (None, "group")])
@pytest.mark.parametrize("bs,length,critic", [(1, 1, True), (8, 7, False), (9, 1000, False), (6, 2047, True),
                                              (6, 2048, False), (5, 2049, True), (70, 129, True)])
def test_padded_advantages(bs, length, critic, levels):
    g = torch.Generator().manual_seed(bs * length)
    lens = torch.randint(1, length + 1, (bs,), generator=g)
    pos = torch.arange(length)[None]
    attn = pos < lens[:, None]
    data = dict(input_ids=torch.zeros(bs, length, dtype=torch.long), attention_mask=attn,
                loss_mask=attn & (pos >= lens[:, None] // 4), logprobs=torch.randn(bs, length, generator=g) * 0.1 - 1,
                rewards=torch.randn(bs, generator=g) * 3)
    if critic:
        data["values"] = torch.randn(bs, length, generator=g)
    norm = Normalization(NormConfig(mean_level=levels[0], std_level=levels[1], group_size=4))
    out = compute_advantages({k: v.to(DEV) for k, v in data.items()}, kl_ctl=0.0, kl_estimator=KLEstimator("k1"),
                             reward_bias=0.5, reward_scaling=2.0, reward_clip=5.0, reward_norm=norm, adv_norm=norm,
                             discount=1.0, gae_lambda=0.95)
    score = torch.clip((data["rewards"] + 0.5) * 2.0, min=-5.0, max=5.0)
    score = N.normalization(score, None, mean_level=levels[0], std_level=levels[1], group_size=4)
    rewards = torch.zeros(bs, length)
    rewards[torch.arange(bs), (lens - 2).clamp(min=0)] = score.float()
    _close(out["tot_rewards"], rewards)
    mask = torch.roll(data["loss_mask"].float(), -1, -1)
    values = data.get("values", torch.zeros(bs, length))
    adv, ret = G.gae_padded(rewards, values, mask, lens == length, 1.0, 0.95)
    _close(out["returns"], ret)
    _close(out["advantages"], N.normalization(adv, mask, mean_level=levels[0], std_level=levels[1], group_size=4))


# a block per row pays for short rows while all blocks are resident at once, and for rows of nearly a tile always
@pytest.mark.parametrize("bs,length,a_block_per_row", [(1024, 100, True), (1025, 100, False), (4096, 64, False),
                                                       (1025, 1791, False), (1025, 1792, True)])
def test_padded_advantages_of_many_rows(monkeypatch, bs, length, a_block_per_row):
    taken = []
    real = actor._token_level_gae_with_row_stats
    monkeypatch.setattr(actor, "_token_level_gae_with_row_stats", lambda *a: taken.append(real(*a)) or taken[-1])
    test_padded_advantages(bs, length, bs % 2 == 0, ("group", "group"))
    assert (taken[0] is not None) == a_block_per_row


@pytest.mark.parametrize("levels", [("group", "group"), ("batch", "batch"), ("batch", "group")])
@pytest.mark.parametrize("lens,group", [([5000], 1), ([4096, 4096, 1], 1), ([300] * 64, 1), ([2048] * 8, 2),
                                        ([17, 4079, 9000, 2, 700, 6000, 300], 3)])
def test_packed_advantages(lens, group, levels):
    g = torch.Generator().manual_seed(sum(lens))
    n = sum(lens)
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32)
    mask = (torch.rand(n, generator=g) > 0.2).float()
    mask[cu[1:].long() - 1] = 0.0
    rewards, values = torch.randn(n, generator=g), torch.randn(n, generator=g)
    norm = Normalization(NormConfig(mean_level=levels[0], std_level=levels[1], group_size=group))
    got, ret, adv = compute_gae_packed_normalized(rewards.to(DEV), values.to(DEV), mask.to(DEV), cu.to(DEV), None, 1.0,
                                                  0.95, norm)
    want, want_ret = G.gae_packed(rewards, values, mask, cu, torch.zeros(len(lens), dtype=torch.bool), 1.0, 0.95)
    _close(adv, want)
    _close(ret, want_ret)
    # the padded form of the oracle: masked rows of the longest sequence
    rows = torch.zeros(len(lens), max(lens))
    row_mask = torch.zeros_like(rows)
    for i, (a, b) in enumerate(zip(cu[:-1].tolist(), cu[1:].tolist())):
        rows[i, : b - a], row_mask[i, : b - a] = want[a:b], mask[a:b]
    normed = N.normalization(rows, row_mask, mean_level=levels[0], std_level=levels[1], group_size=group)
    _close(got, torch.cat([normed[i, :k] for i, k in enumerate(lens)]))


@pytest.mark.parametrize("lambdas", [False, True])
@pytest.mark.parametrize("lens,group", [([2049], 1), ([7000, 3], 1), ([1500, 9000, 100, 2047], 2)])
def test_packed_advantages_without_values(lens, group, lambdas):
    """The C entry point with values = NULL: sequences that go on in the next tiles carry a state without them
    (bitwise what explicit zeros give)."""
    g = torch.Generator().manual_seed(sum(lens))
    n, n_seqs = sum(lens), len(lens)
    lib = _lib.load()
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32).to(DEV)
    mask, rewards = (torch.rand(n, generator=g) > 0.2).float().to(DEV), torch.randn(n, generator=g).to(DEV)
    lam = torch.rand(n_seqs, generator=g).to(DEV) if lambdas else None
    no_eos = torch.arange(n_seqs, device=DEV) % 2 == 0
    first = torch.arange(0, n_seqs + 1, group, device=DEV)
    rows = torch.full((n_seqs // group,), group, device=DEV)
    size = lib.areal_gae_segment_stats_bytes(n, rows.numel())

    def call(values):
        outs = [torch.empty(n, device=DEV) for _ in range(3)]
        scratch = torch.empty(size, dtype=torch.uint8, device=DEV)
        rc = lib.areal_gae_packed_normalized(
            _lib.ptr(rewards), _lib.ptr(values), _lib.ptr(mask), _lib.ptr(cu), _lib.ptr(no_eos), _lib.ptr(lam), n, n_seqs,
            1.0, 0.95, _lib.ptr(first), _lib.ptr(rows), rows.numel(), -1, 2, 2, 1, 1e-5, *[_lib.ptr(o) for o in outs],
            _lib.ptr(scratch), size, _lib.stream_ptr(DEV),
        )
        _lib.check(rc, "areal_gae_packed_normalized")
        return outs

    for got, want in zip(call(None), call(torch.zeros(n, device=DEV))):
        assert torch.equal(got, want)
