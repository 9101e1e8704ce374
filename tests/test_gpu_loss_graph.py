"""A loss call in a captured graph: its results are the graph's own memory and not host memory that
someone else has by the time of a replay, so the statistics read behind a replay are that replay's (one read: the
first is kept)."""

import pytest
import torch

from areal_amd.ppo.actor import grpo_loss_fn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [dict(), dict(use_cispo_loss=True, eps_clip_higher=0.28)])
def test_replayed_statistics(kind):
    dev = torch.device("cuda", 0)
    n = 3000
    g = torch.Generator().manual_seed(0)
    prox = (torch.randn(n, generator=g) * 0.5 - 1).to(dev)
    data = dict(logprobs=prox + 0.1 * torch.randn(n, generator=g).to(dev), prox_logp=prox,
                advantages=torch.randn(n, generator=g).to(dev), loss_mask=(torch.rand(n, generator=g) > 0.2).to(dev))
    lp, ent = torch.empty(n, device=dev).requires_grad_(True), torch.rand(n, generator=g).to(dev)
    inputs = [(prox + 0.1 * torch.randn(n, generator=g).to(dev)) for _ in range(3)]

    def call():
        stats = {}
        loss = grpo_loss_fn(lp, ent, data, eps_clip=0.2, c_clip=None, defer_host_reads=True, stats=stats,
                            stats_mode="reduced", **({"eps_clip_higher": None} | kind))
        return loss, stats["reduction"]

    lp.data.copy_(inputs[0])
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream(dev).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        loss, reduction = call()
    for i, x in enumerate(inputs):
        lp.data.copy_(x)
        want_loss, want = call()
        want = want.results  # the program's own work and a wait for it between the replays
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(loss, want_loss)
        if i == len(inputs) - 1:  # read once, behind the last replay
            assert reduction.results == want
