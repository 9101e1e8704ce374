"""The packing kernels where their layout changes: runs of every length modulo 16 bytes and at every
alignment, totals around a block's 2048 tokens, more tensors than one launch pads, and fills of each
element size; byte for byte against the oracle."""

import pytest
import torch

from areal_amd import _lib
from areal_amd.packing import pack_tensor_dict, pad_packed_tensor_dict, unpack_reorder_pad
from oracle import packing as P

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _to(d):
    return {k: (v.to(DEV) if torch.is_tensor(v) else v) for k, v in d.items()}


def _same(a, b):
    assert a.keys() == b.keys()
    for k in a:
        if torch.is_tensor(b[k]):
            assert a[k].dtype == b[k].dtype and torch.equal(a[k].cpu(), b[k]), k
        else:
            assert a[k] == b[k], k


@pytest.mark.parametrize("lens", [list(range(1, 40)), [1], [15, 1, 16, 17, 31, 33, 5000, 2]])
def test_short_and_unaligned_runs(lens):
    S = max(lens)
    g = torch.Generator().manual_seed(S)
    mask = torch.arange(S)[None] < torch.tensor(lens)[:, None]
    shape = (len(lens), S)
    data = dict(attention_mask=mask, b=torch.randint(0, 255, shape, generator=g).to(torch.uint8),
                h=torch.randint(-99, 99, shape, generator=g).to(torch.int16), f=torch.randn(shape, generator=g),
                odd=torch.randint(0, 255, (*shape, 3), generator=g).to(torch.uint8))
    packed = pack_tensor_dict(_to(data))
    _same(packed, P.pack_tensor_dict(data))
    order = torch.randperm(len(lens), generator=g).tolist()
    for k in ("b", "h", "f", "odd"):
        want = P.unpack_reorder_pad(packed[k].cpu(), lens, order)
        assert torch.equal(unpack_reorder_pad(packed[k], lens, order).cpu(), want), k


@pytest.mark.parametrize("total", [1, 2047, 2048, 2049, 6000])
@pytest.mark.parametrize("extra", [1, 15, 2048, 5000])
@pytest.mark.parametrize("channels", [None, 3])
def test_batch_pad(total, extra, channels):
    g = torch.Generator().manual_seed(total + extra)
    cut = sorted({0, total // 3, total // 2, total})
    cu = torch.tensor(cut, dtype=torch.int32)
    pos = torch.cat([torch.arange(b - a) for a, b in zip(cut[:-1], cut[1:])])
    if channels:
        pos = torch.stack([pos + i for i in range(channels)], dim=1)
    data = dict(cu_seqlens=cu, max_seqlen=max(b - a for a, b in zip(cut[:-1], cut[1:])), position_ids=pos)
    types = [torch.int64, torch.int32, torch.int16, torch.int8, torch.uint8, torch.float32, torch.bfloat16,
             torch.float64, torch.bool, torch.complex128]
    for i, t in enumerate(types):  # with the position ids: two launches
        data[f"t{i}"] = torch.randint(0, 2 if t == torch.bool else 100, (total,), generator=g).to(t)
    for value in (0.0, 3.0):
        want = P.pad_packed_tensor_dict(dict(data), total + extra, value, None)
        got = pad_packed_tensor_dict(_to(data), total + extra, value)
        _same(got[0], want[0])
        assert got[1] == want[1] and torch.equal(got[2].cpu(), want[2])


def test_more_short_rows_than_a_launch_has_blocks(dev):
    """1.2e9 tokens in rows of 12: chunks of five rows are 18.7 million blocks, and a launch takes 2^24 of 256 threads."""
    rows, length = 100_000_000, 12
    padded = torch.randint(0, 255, (rows * length,), dtype=torch.uint8, device=dev)
    packed = torch.zeros_like(padded)
    cu = torch.arange(0, rows * length + 1, length, dtype=torch.int32, device=dev)
    rc = _lib.load().areal_pack_padded(_lib.ptr(padded), _lib.ptr(packed), _lib.ptr(cu), rows, length, 1, rows * length,
                                       _lib.stream_ptr(dev))
    _lib.check(rc, "areal_pack_padded")
    assert torch.equal(packed, padded)
