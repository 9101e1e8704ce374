"""Calls with a small result for the host in a captured graph: a replay, which may come after everybody has let go
of the call's results, writes no host memory, and who still has them reads the replay's."""

import pytest
import torch

from areal_amd import _lib
from areal_amd.functional import fused_lm_head_logprobs_entropy
from areal_amd.ppo.gae import _compute_turn_level_gae, _turn_level_gae

pytestmark = pytest.mark.gpu

T, H, V = 96, 128, 1000


def _capture(dev, call):
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream(dev).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return graph, out


def _lm_head_inputs(dev, hot_row):
    g = torch.Generator().manual_seed(21)
    weight = (torch.randn(V, H, generator=g) * 0.3).bfloat16()
    labels = torch.randint(0, 700, (T,), generator=g)
    hidden = (torch.randn(T, H, generator=g) * 0.5).bfloat16()
    if hot_row:  # far above the estimate of the row's maximum: the saved exponentials are of no use
        hidden[5] = (weight[777].float() * 20.0).bfloat16()
    return hidden.to(dev), weight.to(dev), labels.to(dev), torch.randn(T, generator=g).to(dev)


def _turn_inputs(dev):
    bs, length = 3, 500
    g = torch.Generator().manual_seed(2)
    pos = torch.arange(length, device=dev).expand(bs, length)
    return dict(rewards=torch.randn(bs, length, generator=g).to(dev), values=torch.randn(bs, length, generator=g).to(dev),
                loss_mask=(pos > 20).float(), turn_ids=(pos // 100).to(torch.int32).contiguous(),
                seq_no_eos_mask=torch.zeros(bs, dtype=torch.bool, device=dev), discount=1.0, gae_lambda=0.9)


@pytest.mark.parametrize("what", ["lm_head", "turn gae", "turn gae, not validated"])
def test_replay_leaves_host_memory_alone(dev, what):
    if what == "lm_head":
        hidden, weight, labels, _ = _lm_head_inputs(dev, False)
        hidden.requires_grad_(True)
        call = lambda: fused_lm_head_logprobs_entropy(hidden, weight, labels, save_probs=True)  # noqa: E731
    else:
        inputs = _turn_inputs(dev)
        if what == "turn gae":
            call = lambda: _turn_level_gae(*[inputs[k] for k in ("rewards", "values", "loss_mask", "turn_ids")], False,  # noqa: E731
                                           inputs["seq_no_eos_mask"], 1.0, 0.9, None)
        else:
            call = lambda: _compute_turn_level_gae(**inputs, validate=False)  # noqa: E731
    graph, out = _capture(dev, call)
    del out
    torch.cuda.synchronize()
    # whoever asks for small pinned arrays now gets the memory that was let go
    mine = [torch.full((1,), 12345, dtype=torch.int32).pin_memory() for _ in range(200)]
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert all(int(t) == 12345 for t in mine)


@pytest.mark.parametrize("hot_row", [False, True])
def test_backward_behind_a_replay(dev, hot_row):
    """The forward was captured, its backward runs behind a replay and looks at that replay's status."""
    hidden, weight, labels, grad = _lm_head_inputs(dev, hot_row)
    h, w = hidden.clone().requires_grad_(True), weight.clone().requires_grad_(True)
    want = fused_lm_head_logprobs_entropy(h, w, labels, save_probs=True)
    want.logprobs.backward(grad)
    static = _lm_head_inputs(dev, False)[0].requires_grad_(True)
    v = weight.clone().requires_grad_(True)
    graph, out = _capture(dev, lambda: fused_lm_head_logprobs_entropy(static, v, labels, save_probs=True))
    static.data.copy_(hidden)
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
    assert int(out.logprobs.grad_fn.probs_status.item()) == int(hot_row)
    assert torch.equal(out.logprobs, want.logprobs)
    out.logprobs.backward(grad)
    assert torch.equal(static.grad, h.grad) and torch.equal(v.grad, w.grad)


def test_turn_flags_are_those_of_the_replay(dev):
    inputs = _turn_inputs(dev)
    ids = inputs["turn_ids"]
    graph, (_, _, flags) = _capture(dev, lambda: _turn_level_gae(
        inputs["rewards"], inputs["values"], inputs["loss_mask"], ids, False, inputs["seq_no_eos_mask"], 1.0, 0.9, None))
    for bad in (False, True, False):
        ids[0, 100] = -1 if bad else 1
        graph.replay()
        assert flags.wait() == (5 if bad else 0)  # negative, and lower than the one before


def test_captured_backward_from_saved_exponentials_is_refused(dev):
    """... before anything is queued: the choice between the two modes is the host's."""
    hidden, weight, labels, grad = _lm_head_inputs(dev, False)
    hidden.requires_grad_(True)

    def step(save_probs):
        hidden.grad = None
        out = fused_lm_head_logprobs_entropy(hidden, weight, labels, save_probs=save_probs)
        out.logprobs.backward(grad)
        return hidden.grad

    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        step(True)
        with pytest.raises(_lib.ArealHipError, match="save_probs=False"):
            with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=side):
                step(True)
    torch.cuda.synchronize()
    graph, got = _capture(dev, lambda: step(False))
    graph.replay()
    got = got.clone()
    torch.cuda.synchronize()
    assert torch.equal(got, step(False))


def test_turn_gae_without_validation_takes_no_host_memory(dev):
    """``validate=False``: nobody reads the flags, so no pinned memory is taken and no copy queued for them."""
    inputs = _turn_inputs(dev)
    requests = lambda: torch.cuda.host_memory_stats()["active_requests.allocated"]  # noqa: E731
    want = _compute_turn_level_gae(**inputs)
    torch.cuda.synchronize()
    before = requests()
    got = _compute_turn_level_gae(**inputs, validate=False)
    assert requests() == before
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
