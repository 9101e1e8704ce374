"""The padding that is launched for the total that a batch's shapes suggest (pad_likely in csrc/host.cpp): when it is not
tried, and what becomes of an error in it."""

import pytest
import torch

from areal_amd import _lib
from areal_amd.packing import pad_packed_tensor_dict

pytestmark = pytest.mark.gpu


def _batch(dev, total, **more):
    cu = torch.tensor([0, total // 3, total], dtype=torch.int32, device=dev)
    return dict(cu_seqlens=cu, max_seqlen=total - total // 3, ids=torch.arange(total, device=dev), **more)


@pytest.mark.parametrize("sizes, tried", [([], True), ([2], True), ([3], True), ([2, 3, 1], True), ([4], False), ([900], False), ([1], True), ([2, 900, 7], False)])
def test_not_tried_where_the_shapes_disagree(dev, sizes, tried):
    """One-dimensional tensors of up to an entry a sequence and one more are not counted; any other length leaves it open which
    of them is the total, and a padding for the wrong one is launched and allocated for nothing."""
    data = _batch(dev, 640, **{f"x{i}": torch.ones(n, device=dev) for i, n in enumerate(sizes)})
    for order in (data, dict(reversed(data.items()))):
        assert isinstance(_lib.host().pad_likely(order, order["cu_seqlens"], 1024), tuple) is tried
        got, pad, cu, _ = pad_packed_tensor_dict(order, 1024)
        assert pad == 384 and torch.equal(cu, data["cu_seqlens"])
        assert torch.equal(got["ids"], torch.cat([data["ids"], torch.zeros(384, dtype=torch.int64, device=dev)]))
        assert all(got[k] is data[k] for k in data if k.startswith("x"))
