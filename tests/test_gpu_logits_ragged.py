"""Logits-in kernels at rows of any start and length, either side of the rules on row and block counts."""

import pytest
import torch

from areal_amd.functional import gather_logprobs_entropy
from oracle import logprob as L

pytestmark = pytest.mark.gpu


# 8 elements are a vector of bf16, 4 of fp32; a block of the backward takes 512 vectors; 1024 rows are the
# forward's line between blocks of 1024 and of 256 threads
@pytest.mark.parametrize("rows, vocab, pitch", [
    (3, 1, 1), (5, 7, 7), (5, 8, 11), (4, 15, 15), (3, 2047, 2049), (3, 2049, 2056), (2, 4095, 4097), (2, 4103, 4103),
    (3, 16391, 16396), (1023, 333, 333), (1024, 333, 333), (1025, 37, 41),
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_ragged_rows(dev, rows, vocab, pitch, dtype):
    g = torch.Generator().manual_seed(rows * pitch)
    base = (torch.randn(rows * pitch + 3, generator=g) * 2).to(dtype)
    y = torch.randint(0, vocab, (rows,), generator=g)
    y[0], y[-1] = 0, vocab - 1
    w_lp, w_ent = torch.randn(rows, generator=g), torch.randn(rows, generator=g)
    for start in (0, 1, 3):  # rows of any start, a pitch wider than the row
        x = base[start:start + rows * pitch].view(rows, pitch)[:, :vocab]
        xg = base.to(dev)[start:start + rows * pitch].view(rows, pitch)[:, :vocab].detach().requires_grad_(True)
        lp, ent = gather_logprobs_entropy(xg, y.to(dev), 0.9)
        want_lp, want_ent = L.gather_logprobs_entropy(x, y, 0.9)
        torch.testing.assert_close(lp.cpu(), want_lp, rtol=1e-5, atol=2e-5)
        torch.testing.assert_close(ent.cpu(), want_ent, rtol=1e-5, atol=2e-5)
        ((lp * w_lp.to(dev)).sum() + (ent * w_ent.to(dev)).sum()).backward()
        want = L.logits_backward(x, y, w_lp, w_ent, 0.9)
        tol = dict(rtol=1e-5, atol=2e-5) if dtype == torch.float32 else dict(rtol=1e-2, atol=1e-4)
        torch.testing.assert_close(xg.grad.cpu().float(), want, **tol)
        xg.grad = None
        (gather_logprobs_entropy(xg, y.to(dev), 0.9)[0] * w_lp.to(dev)).sum().backward()
        torch.testing.assert_close(xg.grad.cpu().float(), L.logits_backward(x, y, w_lp, None, 0.9), **tol)


def test_excluded_vocabulary_keeps_its_logprob(dev):
    """Logits of -inf (a masked vocabulary) count nothing, also where a thread meets nothing else."""
    g = torch.Generator().manual_seed(2)
    x = torch.randn(6, 5003, generator=g)
    x[:, 100:4000] = float("-inf")
    y = torch.randint(0, 100, (6,), generator=g)
    lp, _ = gather_logprobs_entropy(x.to(dev), y.to(dev))
    torch.testing.assert_close(lp.cpu(), torch.log_softmax(x, -1)[torch.arange(6), y], rtol=1e-5, atol=2e-5)


# a thread's first elements, its last, the row's edges; one NaN that a thread of its own meets (rows of 5 and 9)
@pytest.mark.parametrize("rows", [3, 1023, 1024])
@pytest.mark.parametrize("vocab", [5, 9, 333, 2051])
@pytest.mark.parametrize("value", [float("-inf"), float("nan"), float("inf")])
def test_logits_that_are_not_finite(dev, value, vocab, rows):
    """As ``torch.log_softmax`` has them, on either side of the forward's line on rows: a NaN or +inf makes the row
    NaN, -inf leaves the log-probabilities of the others alone and the entropy (0 x -inf) NaN."""
    g = torch.Generator().manual_seed(rows + vocab)
    base = torch.randn(rows * vocab + 3, generator=g)
    y = torch.randint(0, vocab, (rows,), generator=g)
    for start in (0, 1, 3):
        x = base[start:start + rows * vocab].view(rows, vocab).clone()
        for i in range(0, rows, 2):
            x[i, (7 * i) % vocab] = value
            if value == float("-inf") and i % 4 == 0:  # whole threads of nothing else
                x[i, : vocab - 2] = value
        xg = base.to(dev)[start:start + rows * vocab].view(rows, vocab)
        xg.copy_(x.to(dev))
        lp, ent = gather_logprobs_entropy(xg, y.to(dev))
        want_lp, want_ent = L.gather_logprobs_entropy(x, y)
        torch.testing.assert_close(lp.cpu(), want_lp, rtol=1e-5, atol=2e-5, equal_nan=True)
        torch.testing.assert_close(ent.cpu(), want_ent, rtol=1e-5, atol=2e-5, equal_nan=True)


# bytes either side of the rule on how many rows the forward keeps in the memory-side cache for the backward: none of a
# batch left out, a few, and more than half of one above 512 MB
@pytest.mark.parametrize("rows", [1046, 1047, 1100, 2200])
def test_rows_kept_for_the_backward(dev, rows):
    """Same bits whether a row is kept or not (a forward without a gradient keeps none); against 64 bits either side of the line."""
    vocab = 128256
    g = torch.Generator(device=dev).manual_seed(rows)
    x = (torch.randn(rows, vocab, generator=g, device=dev) * 2).bfloat16()
    y = torch.randint(0, vocab, (rows,), generator=g, device=dev)
    w = torch.randn(rows, generator=g, device=dev)
    xg = x.detach().requires_grad_(True)
    lp, ent = gather_logprobs_entropy(xg, y)
    with torch.no_grad():
        plain_lp, plain_ent = gather_logprobs_entropy(x, y)
    assert torch.equal(lp, plain_lp) and torch.equal(ent, plain_ent)
    (lp * w).sum().backward()
    size = 2 * vocab
    line = ((256 if rows * size <= 512 << 20 else 320) << 20) // size
    at = sorted({i for i in (0, 1, line - 1, line, rows - 2, rows - 1) if 0 <= i < rows})
    logp = torch.log_softmax(x[at].double(), -1)
    pick = (torch.arange(len(at), device=dev), y[at])
    torch.testing.assert_close(lp[at].double(), logp[pick], rtol=1e-5, atol=2e-5)
    torch.testing.assert_close(ent[at].double(), -(logp.exp() * logp).sum(-1), rtol=1e-5, atol=2e-5)
    want = -logp.exp() * w[at, None].double()
    want[pick] += w[at].double()
    torch.testing.assert_close(xg.grad[at].double(), want, rtol=1e-2, atol=1e-6)


@pytest.mark.parametrize("rows", [1046, 1047, 3678, 3680])
def test_the_rows_either_side_of_those_kept(dev, rows):
    """The last 256 MB of the rows, or 512 of more than 900, are read without the non-temporal hint when a gradient is wanted: the
    same bits as without one, on rows either side of the line; their gradient against 64 bits."""
    vocab = 128256
    g = torch.Generator(device=dev).manual_seed(rows)
    x = (torch.randn(rows, vocab, generator=g, device=dev) * 2).bfloat16().requires_grad_(True)
    y = torch.randint(0, vocab, (rows,), generator=g, device=dev)
    w = torch.randn(rows, generator=g, device=dev)
    lp, ent = gather_logprobs_entropy(x, y)
    with torch.no_grad():
        plain_lp, plain_ent = gather_logprobs_entropy(x.detach(), y)
    assert torch.equal(lp, plain_lp) and torch.equal(ent, plain_ent)
    (lp * w).sum().backward()
    size = 2 * vocab
    line = rows - ((256 if rows * size <= 900 << 20 else 512) << 20) // size
    at = sorted({i for i in (0, line - 1, line, line + 1, rows - 1) if 0 <= i < rows})
    logp = torch.log_softmax(x.detach()[at].double(), -1)
    pick = (torch.arange(len(at), device=dev), y[at])
    torch.testing.assert_close(lp[at].double(), logp[pick], rtol=1e-5, atol=2e-5)
    want = -logp.exp() * w[at, None].double()
    want[pick] += w[at].double()
    torch.testing.assert_close(x.grad[at].double(), want, rtol=1e-2, atol=1e-6)
