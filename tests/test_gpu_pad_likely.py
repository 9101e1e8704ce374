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


@pytest.fixture
def little_memory(dev):
    """A quarter GiB for what is allocated from here on."""

    def limit():
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        room = torch.cuda.memory_reserved(dev) + (256 << 20)
        torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(dev).total_memory, dev)

    yield limit
    torch.cuda.set_per_process_memory_fraction(1.0, dev)


def test_out_of_memory_is_reported_once(dev, little_memory):
    """A padding that does not fit is not tried a second time on the way for other batches."""
    data = _batch(dev, 1000)
    little_memory()
    before = torch.cuda.memory_stats(dev)["num_ooms"]
    with pytest.raises(torch.OutOfMemoryError):
        pad_packed_tensor_dict(data, 1 << 27)
    assert torch.cuda.memory_stats(dev)["num_ooms"] == before + 1
    assert pad_packed_tensor_dict(data, 2000)[1] == 1000


def test_a_wrong_padding_that_does_not_fit(dev, little_memory):
    """The one-dimensional tensors are no token tensors: only the padding that nobody asked for is too large."""
    data = _batch(dev, 1000, **{f"table{i}": torch.ones(10 << 20, device=dev) for i in range(3)})
    data["ids"] = data["ids"].view(1, -1)
    little_memory()
    got, pad, _, _ = pad_packed_tensor_dict(data, 30 << 20)
    assert pad == (30 << 20) - 1000 and all(got[k] is data[k] for k in data if k.startswith("table"))
    torch.cuda.set_per_process_memory_fraction(1.0, dev)
    assert torch.equal(got["ids"], torch.nn.functional.pad(data["ids"][0], (0, pad)))
