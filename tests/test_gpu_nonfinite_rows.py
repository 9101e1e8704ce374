"""Rows with a NaN or infinite logit that is not the label's: the log-probability is that of ``torch.log_softmax``
(NaN for the whole row), from every sweep that makes one, and never the 0 of a certain token.

A weight row of NaN makes one logit of every token NaN; one with an infinite entry makes it +inf or -inf by the sign of the
hidden value (-inf counts nothing). One such row, and 500 in a row: whole tiles without another logit. Finite results: |error| <= 2^-20 of the largest |logit| + 2^-18, as for fp32 sums."""

import pytest
import torch

from areal_amd.engine import compute_logprobs
from areal_amd.functional import fused_lm_head_logprobs_entropy

pytestmark = pytest.mark.gpu


# 128: the hand-scheduled sweeps, 72: the generic one; 1600 ends in a last tile that overlaps its predecessor
@pytest.mark.parametrize("T,H,V", [(140, 128, 1536), (140, 128, 1600), (70, 72, 600)])
@pytest.mark.parametrize("entry", [float("nan"), float("inf")])
@pytest.mark.parametrize("rows", [1, 500])
@pytest.mark.parametrize("sweep", ["logprobs_only", "no_grad", "saved", "recompute"])
def test_bad_weight_rows(dev, sweep, rows, entry, T, H, V):
    g = torch.Generator().manual_seed(V)
    hidden = torch.randn(T, H, generator=g).bfloat16()
    weight = (torch.randn(V, H, generator=g) * 0.1).bfloat16()
    bad = V - 7
    weight[bad + 1 - rows:bad + 1, 0] = entry
    labels = torch.randint(0, V, (T,), generator=g)
    labels[5], labels[6] = bad, bad
    x = hidden.float() @ weight.float().t()
    want = torch.log_softmax(x.double(), -1).gather(1, labels[:, None])[:, 0]
    assert not want.isfinite().all()
    h, w, y = hidden.to(dev), weight.to(dev), labels.to(dev)
    if sweep == "logprobs_only":
        got = compute_logprobs(h, w, dict(rolled_input_ids=y))
    elif sweep == "no_grad":
        with torch.no_grad():
            got = fused_lm_head_logprobs_entropy(h, w, y).logprobs
    else:
        got = fused_lm_head_logprobs_entropy(h.requires_grad_(True), w, y, save_probs=sweep == "saved").logprobs.detach()
    got = got.cpu().double()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isfinite(), want.isfinite())
    ok = want.isfinite()
    tol = 2.0 ** -20 * x[x.isfinite()].abs().max().item() + 2.0 ** -18
    assert not ok.any() or (got[ok] - want[ok]).abs().max().item() <= tol
