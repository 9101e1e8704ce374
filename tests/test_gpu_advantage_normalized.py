"""Advantages that come out normalised from the launch that makes them (areal_advantages_normalized) against the two
launches it replaces (areal_advantages_row_stats, areal_group_norm_from_row_stats): the same scan and the same sums added up in the
same order, so the same bits.

Rows around the tile and up to the longest it takes, groups of one row, of the most rows it takes, ragged ones; a group
without a masked token and a batch without any; advantages that are not finite. With no time to wait every row whose
group is not complete yet leaves its normalisation to the group's last, which has to give the same bits."""

import ctypes

import pytest
import torch

from areal_amd import _lib
from areal_amd.config import NormConfig
from areal_amd.data import KLEstimator, Normalization
from areal_amd.ppo.actor import compute_advantages

pytestmark = pytest.mark.gpu


def _inputs(dev, bs, L, critic, ref):
    g = torch.Generator().manual_seed(31 * bs + L)
    lens = torch.randint(1, L + 1, (bs,), generator=g)
    lens[0] = L
    attn = torch.arange(L)[None] < lens[:, None]
    normal = lambda: torch.randn(bs, L, generator=g)  # noqa: E731
    return dict(loss=(attn & (torch.rand(bs, L, generator=g) > 0.3)).to(dev), attn=attn.to(dev), logp=(normal() - 1).to(dev),
                ref=(normal() - 1).to(dev) if ref else None, values=normal().to(dev) if critic else None,
                rewards=torch.randn(bs, generator=g).to(dev))


def _both(dev, x, offsets, levels, unbiased, wait_us, eps=1e-5, fill=0):
    """(two launches, one launch): normalised advantages and the other outputs."""
    lib = _lib.load()
    bs, L = x["logp"].shape
    rows = torch.tensor([(b - a) for a, b in zip(offsets[:-1], offsets[1:])], device=dev)
    off = torch.tensor(offsets, device=dev) * L
    most = int(rows.max())
    res = []
    for fused in (False, True):
        f32 = lambda: torch.full((bs, L), float("nan"), device=dev)  # noqa: E731
        lm, old, kl, tot, adv, ret = (f32() for _ in range(6))
        ref = x["ref"].clone() if x["ref"] is not None else None
        lens, eos = torch.empty(bs, dtype=torch.int64, device=dev), torch.empty(bs, dtype=torch.bool, device=dev)
        p, s = _lib.ptr, _lib.stream_ptr(dev)
        args = [p(x["rewards"]), 1, 0.1, 1.5, 2.0, None, None, 0, -1, 0, 0, 0, 0.0, p(x["loss"]), p(x["attn"]), p(x["logp"]),
                p(ref), p(x["values"]), bs, L, 1, 1, 1, 0, int(ref is not None), 0.1, 0.99, 0.95, p(lm), p(old), p(kl),
                p(tot), p(lens), p(eos), p(adv), p(ret)]
        if fused:
            spec = _lib.GroupNormSpec(off.data_ptr(), len(rows), most, -1, *levels, 0, unbiased, wait_us, eps)
            nbytes = lib.areal_advantages_normalized_workspace_bytes(bs)
            ws = torch.full((nbytes,), fill, dtype=torch.uint8, device=dev)
            _lib.check(lib.areal_advantages_normalized(*args, ctypes.byref(spec), p(ws), nbytes, s), "normalized")
        else:
            sums = torch.empty(5, bs, dtype=torch.float64, device=dev)
            _lib.check(lib.areal_advantages_row_stats(*args, p(sums), s), "row_stats")
            out = f32()
            _lib.check(lib.areal_group_norm_from_row_stats(
                p(adv), p(lm), bs, L, p(off), p(rows), len(rows), most * L, -1, *levels, unbiased, eps, p(sums), p(out), s),
                "from_row_stats")
            adv = out
        torch.cuda.synchronize()
        res.append((adv, ret, lm, old, kl, tot, lens, eos))
    return res


def _same(a, b):
    for x, y in zip(a, b):
        assert torch.equal(x.nan_to_num(7.5), y.nan_to_num(7.5))
        assert torch.equal(x.isnan(), y.isnan())


@pytest.mark.parametrize("wait_us", [-1, 0])
@pytest.mark.parametrize("L", [1, 255, 1793, 2048, 2049, 6143, 8191, 8192])
@pytest.mark.parametrize("offsets", [[0, 1], [0, 1, 5, 8], [0, 64], [0, 3, 67, 68, 100]])
def test_same_bits_as_two_launches(dev, offsets, L, wait_us):
    bs = offsets[-1]
    x = _inputs(dev, bs, L, critic=bs != 8, ref=bs != 64)
    if len(offsets) > 2:
        x["loss"][offsets[1]:offsets[2]] = False  # a group without a masked token
    levels = [(2, 2), (0, 2), (2, 0)][bs % 3]
    _same(*_both(dev, x, offsets, levels, bs % 2, wait_us))


@pytest.mark.parametrize("wait_us", [-1, 0])
def test_nothing_active_and_not_finite(dev, wait_us):
    x = _inputs(dev, 12, 2500, True, True)
    x["values"][5, 17] = float("inf")
    x["values"][9, 2000] = float("nan")
    _same(*_both(dev, x, [0, 4, 8, 12], (2, 2), 1, wait_us))
    x["loss"].zero_()
    _same(*_both(dev, x, [0, 4, 8, 12], (2, 2), 1, wait_us))


def test_many_groups_with_rows_that_leave(dev):
    """More rows than are on the chip at once, none of which waits."""
    x = _inputs(dev, 4096, 1800, True, False)
    _same(*_both(dev, x, list(range(0, 4097, 16)), (2, 2), 1, 0))


@pytest.mark.parametrize("fill", [0, 0, 64, 255])
def test_sums_of_few_bits(dev, fill):
    """Counts and sums that are small integers, told from what the workspace held before."""
    x = _inputs(dev, 1024, 1024, False, False)
    x["loss"].fill_(True)
    x["attn"].fill_(True)
    x["logp"].fill_(-1.0)
    x["rewards"].copy_((x["rewards"] > 0).float())
    _same(*_both(dev, x, list(range(0, 1025, 16)), (2, 2), 1, -1, fill=fill))


@pytest.mark.parametrize("change", ["batch", "tail", "long group", "long row", "leave one out"])
def test_what_it_does_not_take(dev, change):
    lib = _lib.load()
    fake = 0x10000  # never dereferenced: the rules come first
    spec = _lib.GroupNormSpec(fake, 2, 64, -1, 2, 2, 0, 1, -1, 1e-5)
    if change == "batch":
        spec.mean_level = 1
    elif change == "tail":
        spec.tail_group = 1
    elif change == "long group":
        spec.max_group_rows = 65
    elif change == "leave one out":
        spec.leave_one_out = 1
    L = 8193 if change == "long row" else 8192
    rc = lib.areal_advantages_normalized(
        fake, 1, 0.0, 1.0, 20.0, None, None, 0, -1, 0, 0, 0, 0.0, fake, fake, fake, None, None, 66, L, 0, 1, 0, 0, 0, 0.1, 0.99,
        0.95, fake, fake, fake, fake, fake, fake, fake, fake, ctypes.byref(spec), fake, 1 << 20, None)
    assert rc == _lib.ERR_UNSUPPORTED


def test_captured_call_takes_two_launches(dev):
    """A graph's replays would all carry the captured call's number: such a call is made of two launches, and every replay
    gives what an eager call gives."""
    x = _inputs(dev, 32, 1000, True, True)
    norm = Normalization(NormConfig(mean_level="group", std_level="group", group_size=8))
    data = dict(input_ids=torch.zeros(32, 1000, dtype=torch.long, device=dev), attention_mask=x["attn"], loss_mask=x["loss"],
                logprobs=x["logp"], rewards=x["rewards"], values=x["values"])
    call = lambda: compute_advantages(dict(data), kl_ctl=0.1, kl_estimator=KLEstimator("k1"), adv_norm=norm,  # noqa: E731
                                      discount=0.99, gae_lambda=0.95)["advantages"]
    want = [call().clone()]
    side = torch.cuda.Stream(dev)
    with torch.cuda.stream(side):
        call()
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = call()
    first = x["rewards"].clone()
    for k in range(3):
        x["rewards"].copy_(first * (k + 1))
        want = call().clone()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want), k
