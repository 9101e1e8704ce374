"""A host that has to know a small result of the GPU's waits for the call that makes it, and not for what was
queued behind that call: the lm_head's backward returns once its forward has finished, deferred results of a
loss call can be read while later work runs. All at sizes where the GPU is busy for milliseconds."""

import functools
import math

import pytest
import torch

from areal_amd.config import NormConfig, RejectionSamplingConfig
from areal_amd.data import KLEstimator, Normalization
from areal_amd.functional import StatReduction, fused_lm_head_logprobs_entropy, gather_logprobs_entropy
from areal_amd.ppo import actor
from areal_amd.ppo.actor import compute_advantages, grpo_loss_fn

pytestmark = pytest.mark.gpu


def _busy(dev, products):
    """Work for about ``products`` milliseconds."""
    a = torch.ones(8192, 8192, dtype=torch.bfloat16, device=dev)
    out = torch.empty_like(a)

    def queue():
        for _ in range(products):
            torch.mm(a, a, out=out)
        done = torch.cuda.Event()
        done.record()
        return done

    queue().synchronize()  # (the library's own preparations)
    return queue


def _loss_data(dev, n, seed):
    g = torch.Generator().manual_seed(seed)
    prox = (torch.randn(n, generator=g) * 0.1 - 12).to(dev)
    return dict(logprobs=prox + (torch.randn(n, generator=g) * 0.1).to(dev), prox_logp=prox,
                advantages=torch.randn(n, generator=g).to(dev), loss_mask=(torch.rand(n, generator=g) > 0.2).to(dev))


LOSS = functools.partial(grpo_loss_fn, eps_clip=0.2, eps_clip_higher=None, c_clip=None, stats_mode="reduced",
                         defer_host_reads=True, rejection_sampling=RejectionSamplingConfig(
                             level="token", action="mask", metric="ratio", lower=0.5, upper=2.0))


def test_backward_returns_when_the_forward_has_finished(dev):
    T, H, V = 8192, 2048, 151936  # forward about 4 ms, backward about 8
    g = torch.Generator(device=dev).manual_seed(3)
    h = torch.randn(T, H, generator=g, device=dev, dtype=torch.bfloat16).requires_grad_(True)
    w = (torch.randn(V, H, generator=g, device=dev, dtype=torch.bfloat16) * 0.02).requires_grad_(True)
    labels = torch.randint(0, V, (T,), generator=g, device=dev)
    data = _loss_data(dev, T, 3)
    later = _busy(dev, 1)

    def step():
        h.grad = w.grad = None
        stats = {}
        out = fused_lm_head_logprobs_entropy(h, w, labels, save_probs=True)
        loss = LOSS(out.logprobs, out.entropy, data, stats=stats)
        loss.backward()
        return loss, stats

    step()  # warm-up: allocator and pinned-memory pools
    torch.cuda.synchronize()
    torch.cuda.set_sync_debug_mode("error")
    try:
        loss, stats = step()
        done = later()
        assert not done.query()  # the backward and what the host queued behind it are still to be done
    finally:
        torch.cuda.set_sync_debug_mode("default")
    results = stats["reduction"].results
    torch.cuda.synchronize()
    assert results["new_logp"]["count"] == float(data["loss_mask"].sum())


def test_deferred_results_are_read_while_later_work_runs(dev):
    n = 8192
    data = _loss_data(dev, n, 4)
    lp, entropy = data["prox_logp"].clone().requires_grad_(True), torch.zeros(n, device=dev)
    before, later = _busy(dev, 5), _busy(dev, 60)
    before()
    stats = {}
    LOSS(lp, entropy, data, stats=stats)
    done = later()
    assert float(stats["scalar/n_valid_tokens"]) == float(stats["reduction"].results["new_logp"]["count"])
    assert not done.query()
    done.synchronize()


def test_turn_ids_are_checked_without_waiting_for_the_normalisation(dev):
    bs, length = 4, 512
    pos = torch.arange(length, device=dev).expand(bs, length)
    data = dict(input_ids=torch.zeros(bs, length, dtype=torch.long, device=dev),
                attention_mask=torch.ones(bs, length, dtype=torch.bool, device=dev),
                loss_mask=pos > 10, logprobs=torch.zeros(bs, length, device=dev), rewards=torch.ones(bs, device=dev),
                turn_ids=(pos // 100).to(torch.int32).contiguous())
    norm = Normalization(NormConfig(mean_level="batch", std_level="batch"))
    before, later = _busy(dev, 5), _busy(dev, 60)
    done = []

    def adv_norm(*args, **kwargs):
        out = norm(*args, **kwargs)
        done.append(later())
        return out

    call = functools.partial(compute_advantages, kl_ctl=0.0, kl_estimator=KLEstimator("k1"), discount=1.0,
                             gae_lambda=0.9, gae_timestep_unit="turn")
    call(dict(data), adv_norm=norm)  # (the groups' tables are made once)
    torch.cuda.synchronize()
    before()
    call(dict(data), adv_norm=adv_norm)
    assert not done[0].query()
    done[0].synchronize()


@pytest.mark.parametrize("options", [dict(), dict(defer_host_reads=False), dict(use_sapo_loss=True, rejection_sampling=None)])
def test_statistics_do_not_hold_the_logits(dev, options, monkeypatch):
    """A reduction keeps the entropies, read or not, but not the graph with the logits behind them."""
    n, vocab = 512, 32768
    data = _loss_data(dev, n, 5)
    labels = torch.zeros(n, dtype=torch.long, device=dev)

    kept = []

    class Kept(StatReduction):
        def __init__(self, *args, **kwargs):
            super().__init__(*args, **kwargs)
            kept.append(self)

    monkeypatch.setattr(actor, "StatReduction", Kept)

    def step():
        logits = torch.zeros(n, vocab, device=dev, requires_grad=True)
        logp, entropy = gather_logprobs_entropy(logits, labels)
        LOSS(logp, entropy, data, stats={}, **options)

    before = torch.cuda.memory_allocated(dev)
    step()
    assert torch.cuda.memory_allocated(dev) - before < 4 * n * vocab
    assert kept[0].results["entropy"]["avg"] == pytest.approx(math.log(vocab), rel=1e-5)


def test_an_entropy_is_asked_for(dev):
    data = _loss_data(dev, 64, 6)
    with pytest.raises(AttributeError):
        LOSS(data["prox_logp"].clone().requires_grad_(True), None, data, stats={})
