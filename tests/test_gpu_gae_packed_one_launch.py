"""Packed GAE and the normalisation of its advantages in one launch (areal_gae_packed_normalized_ex) against the two launches
it replaces (areal_gae_packed_normalized): the same scan, so the same bits of advantages and returns. A group's sums are
added up in fp64 in another order (2^-52 a term, a few thousand of them at most), after which mean and deviation may round to the fp32
neighbour: 2^-23 of each, so |difference| <= 2^-22 (|x| + |mean|) / deviation, with the mean below the largest |x|.

Groups inside a tile, over many tiles, empty ones, more groups in a tile than a block has waves; sequences without
tokens and longer than many tiles; tokens before the first and behind the last sequence; masks that are not 0 or 1, a
group without a masked token, advantages that are not finite. With no time to wait every segment of a group that is not
complete yet is left to the group's last wave, which has to give the same."""

import pytest
import torch

from areal_amd import _lib

pytestmark = pytest.mark.gpu


def _took_one_launch(ws, n, cu, first):
    """Every tile's flag of each of its groups holds the call's number."""
    tiles, groups = -(-n // 2048), first.numel() - 1
    flags = ws.view(torch.int64)[8 * (tiles + groups) : 9 * (tiles + groups)].cpu()
    slots = []
    for g, (a, b) in enumerate(zip(cu[first[:-1]].tolist(), cu[first[1:]].tolist())):
        if a < b:
            slots += [k + g for k in range(a // 2048, (b - 1) // 2048 + 1)]
    assert len(set(flags[slots].tolist())) == 1


def _run(dev, lens, sizes, levels, wait_us, *, unbiased=1, critic=True, lam=None, mask="binary", around=(0, 0), bad=None, fill=0):
    lib = _lib.load()
    g = torch.Generator().manual_seed(len(lens) + sum(lens))
    cu = torch.tensor([around[0]] + lens).cumsum(0).to(torch.int32)
    n, n_seqs = int(cu[-1]) + around[1], len(lens)
    m = (torch.rand(n, generator=g) > 0.4).float()
    if mask == "ones":
        m.fill_(1.0)
    if mask == "weights":
        m *= 0.25 + torch.rand(n, generator=g)
    first = torch.tensor([0] + sizes).cumsum(0)
    if mask == "sparse":
        m = (torch.rand(n, generator=g) > 0.999).float()
    if mask == "silent group":
        m[cu[first[1]]:cu[first[2]]] = 0
    r, v = torch.randn(n, generator=g), torch.randn(n, generator=g)
    if bad is not None:
        r[bad], m[bad] = float("inf"), 1.0
    no_eos = (torch.rand(n_seqs, generator=g) > 0.5).to(dev)
    lam_seq = torch.rand(n_seqs, generator=g).to(dev) if lam else None
    x = [t.to(dev) for t in (r, v, m, cu, first, torch.tensor(sizes))]
    p, s = _lib.ptr, _lib.stream_ptr(dev)
    res = []
    for fused in (False, True):
        adv, ret, out = (torch.full((n,), 7.5, device=dev) for _ in range(3))
        head = [p(x[0]), p(x[1]) if critic else None, p(x[2]), p(x[3]), p(no_eos), p(lam_seq), n, n_seqs, 0.99, 0.95, p(x[4]), p(x[5]),
                len(sizes)]
        if fused:
            nbytes = lib.areal_gae_packed_normalized_workspace_bytes(n, len(sizes))
            ws = torch.full((nbytes,), fill, dtype=torch.uint8, device=dev)
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            _lib.check(lib.areal_gae_packed_normalized_ex(*head, max(sizes), -1, *levels, unbiased, 1e-5, wait_us, p(adv), p(ret),
                                                          p(out), p(ws), nbytes, s), "ex")
            end.record()
        else:
            nbytes = lib.areal_gae_segment_stats_bytes(n, len(sizes))
            ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
            _lib.check(lib.areal_gae_packed_normalized(*head, -1, *levels, unbiased, 1e-5, p(adv), p(ret), p(out), p(ws), nbytes, s),
                       "two launches")
        torch.cuda.synchronize()
        res.append((out, adv, ret))
    _took_one_launch(ws, n, cu, first)
    for k, (a, b) in enumerate(zip(*res)):
        assert torch.equal(a.isnan(), b.isnan())
        a, b = a.nan_to_num(3.25), b.nan_to_num(3.25)
        if k == 0:
            assert (a - b).abs().max().item() <= 2.0 ** -21 * a.abs().max().item()
        else:
            assert torch.equal(a, b)
    if mask == "sparse":
        want = _recurrence(r, v if critic else torch.zeros(n), m, cu, no_eos.cpu(), lam_seq.cpu() if lam else torch.full((n_seqs,), 0.95))
        # masked tokens alone change the state, and each takes the error before it by 0.99 lambda < 0.95: 20 tokens' worth
        # stays, of at most 24 roundings each (8 tokens, 6 steps of the wave's tree, two operations a step)
        assert (res[1][1].cpu().double() - want).abs().max().item() <= 20 * 24 * 2.0 ** -24 * want.abs().max().item()
    return begin.elapsed_time(end) * 1e3


def _recurrence(r, v, m, cu, no_eos, lam):
    """Advantages in fp64, token by token."""
    r, v, m, ends = r.double().tolist(), v.double().tolist(), m.double().tolist(), cu.tolist()
    want = torch.zeros(len(r), dtype=torch.float64)
    for s, (a, b) in enumerate(zip(ends, ends[1:])):
        c, adv, nv = 0.99 * float(lam[s]), 0.0, 0.0
        for t in range(b - 1, a - 1, -1):
            if t == b - 1:
                nv = v[t] if no_eos[s] else 0.0
            else:
                adv, nv = (c * m[t] + 1 - m[t]) * adv + m[t] * (0.99 * nv + r[t] - v[t]), (1 - m[t]) * nv + m[t] * v[t]
            want[t] = adv
    return want


def _lens(n, mean, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.exp(torch.randn(n, generator=g) * 0.8) * mean * 0.73).long().clamp(min=1).tolist()


@pytest.mark.parametrize("wait_us", [-1, 0])
@pytest.mark.parametrize("case", range(8))
def test_same_bits_as_two_launches(dev, case, wait_us):
    lens, sizes, options = [
        (_lens(64, 700, 1), [4] * 16, dict()),
        (_lens(96, 60, 2), [8] * 12, dict(unbiased=0)),                       # several groups in a tile
        (_lens(240, 90, 3), [3, 1, 5, 7] * 15, dict(critic=False)),           # more of them than waves
        (_lens(48, 5000, 4), [16] * 3, dict(lam=True)),                       # groups and sequences of many tiles
        ([2048] * 8 + [0, 1, 4096, 0, 2047, 2049, 0, 0], [4, 4, 2, 2, 2, 2], dict(mask="silent group")),
        (_lens(32, 1500, 6), [8, 8, 0, 8, 0, 8], dict(mask="weights")),
        (_lens(20, 900, 7), [10, 10], dict(around=(37, 5000))),
        (_lens(30, 1200, 8), [6] * 5, dict(bad=5000)),
    ][case]
    levels = [(2, 2), (0, 2), (2, 0), (0, 0)][case % 4]
    _run(dev, lens, sizes, (2, 2), wait_us, **options)
    _run(dev, lens, sizes, levels, wait_us, **options)


@pytest.mark.parametrize("wait_us", [-1, 0])
@pytest.mark.parametrize("case", range(5))
def test_state_carried_over_whole_tiles(dev, case, wait_us):
    """Sequences over 0, 1, 16, 17 and 40 whole tiles, whose maps come from their blocks 16 tiles at a time; as many sequences
    and groups as fit a block's memory and one more of each. One token in 1000 is masked in, so the state goes far."""
    long = [40 * 2048 + 5, 3, 17 * 2048, 18 * 2048 + 1, 0, 1, 2047, 2048, 2049, 3 * 2048, 4095, 5, 0, 1, 17 * 2048 + 2047, 9]
    lens, sizes, options = [
        (long, [8, 8], dict()),
        (long, [8, 8], dict(lam=True, around=(37, 5000))),
        (long[::-1], [8, 8], dict(critic=False)),
        ([120] * 2047 + [30000], [2] * 1023 + [1, 1], dict()),
        ([30000] + [120] * 2048, [2] * 1023 + [3], dict()),
    ][case]
    _run(dev, lens, sizes, (2, 2), wait_us, mask="sparse", **options)


@pytest.mark.parametrize("wait_us", [-1, 0])
@pytest.mark.parametrize("case", range(6))
def test_more_sequences_than_a_block_holds(dev, case, wait_us):
    """Above 2048 sequences a wave searches for them, and what it finds tells the groups while these fit (up to 1024): ends of
    more than 64 sequences in a tile, more sequences in a tile than the block's memory holds, empty groups, tiles before the
    first and behind the last sequence."""
    lens, sizes, options = [
        ([120] * 2049, [3] * 683, dict(around=(37, 5000))),
        ([200] * 2100, [2, 1] * 700, dict(around=(4100, 5000), lam=True)),            # more groups than the block holds
        (_lens(3000, 40, 11), [16, 0, 8] * 125, dict()),
        ([0] * 2500 + [700] * 30 + [0] * 2500 + [1500], [1, 2499, 30, 2500, 1], dict()),
        ([1] * 4200 + [9000] + [1] * 63 + [2048] * 2, [100] * 42 + [66], dict(critic=False)),
        (_lens(4097, 60, 12), [17] * 241, dict()),
    ][case]
    _run(dev, lens, sizes, (2, 2), wait_us, mask="sparse", **options)


@pytest.mark.parametrize("wait_us", [-1, 0])
def test_more_tiles_than_the_chip_holds(dev, wait_us):
    _run(dev, _lens(4800, 700, 9), [4] * 1200, (2, 2), wait_us)


@pytest.mark.parametrize("place", [0, 1600, 3200])
def test_a_group_longer_than_an_xcd_holds(dev, place):
    """More tiles than the chip holds, 195 of them of one group, 128 of which are on an XCD at once: the others have to start
    before the time is up that a tile waits at most, here a millisecond (all of the call takes about 0.2)."""
    lens = _lens(3200, 700, 10)
    lens[place:place] = [100000] * 4
    for _ in range(2):  # (the first one loads the kernels)
        us = _run(dev, lens, [4] * 801, (2, 2), 1000)
    assert us < 900


@pytest.mark.parametrize("fill", [0, 0, 0, 64, 255])
def test_counts_of_few_bits(dev, fill):
    """Whole tiles of masked tokens and small integers make sums with hardly a bit set, which have to be told from
    what the workspace held before, however many of an entry's words have arrived."""
    _run(dev, [2048] * 256 + [1500] * 512, [16] * 48, (2, 2), -1, critic=False, mask="ones", fill=fill)


def test_short_groups(dev):
    for n in (1, 2, 7, 8, 9, 255):
        _run(dev, [n, 600], [1, 1], (2, 2), -1)


def test_captured_call_takes_two_launches(dev):
    """A graph's replays would all carry the captured call's number: they run the two launches and see new inputs."""
    from areal_amd.config import NormConfig
    from areal_amd.data import Normalization
    from areal_amd.ppo.gae import compute_gae_packed_normalized

    g = torch.Generator().manual_seed(0)
    cu = torch.arange(0, 33 * 500, 500, dtype=torch.int32, device=dev)
    r, v, m = (torch.randn(16000, generator=g).to(dev) for _ in range(3))
    m = (m > 0).float()
    norm = Normalization(NormConfig(mean_level="group", std_level="group", group_size=8))
    call = lambda: compute_gae_packed_normalized(r, v, m, cu, None, 1.0, 0.95, norm)  # noqa: E731
    side = torch.cuda.Stream(dev)
    with torch.cuda.stream(side):
        call()
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = call()
    for k in range(3):
        r.add_(v, alpha=0.3)
        want = [t.clone() for t in call()]
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want)), k


@pytest.mark.parametrize("groups", [1, 2, 3, 4])
def test_a_wave_s_map_lies_in_one_line(dev, groups):
    """Whatever the numbers of tiles and groups: six words at the start of a line of 64 bytes, so that a map leaves and comes in
    one piece."""
    lib = _lib.load()
    lens = [5 * 2048 + 7] * groups
    n = sum(lens)
    cu = torch.tensor([0] + lens, device=dev).cumsum(0).to(torch.int32)
    first, rows = torch.arange(groups + 1, device=dev), torch.ones(groups, dtype=torch.int64, device=dev)
    x = [torch.randn(n, device=dev) for _ in range(2)] + [torch.ones(n, device=dev)]
    out = [torch.empty(n, device=dev) for _ in range(3)]
    nbytes = lib.areal_gae_packed_normalized_workspace_bytes(n, groups)
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    assert ws.data_ptr() % 256 == 0
    p = _lib.ptr
    _lib.check(lib.areal_gae_packed_normalized_ex(*map(p, x), p(cu), None, None, n, groups, 0.99, 0.95, p(first), p(rows), groups, 1, -1,
                                                  2, 2, 1, 1e-5, -1, *map(p, out), p(ws), nbytes, _lib.stream_ptr(dev)), "ex")
    tiles = -(-n // 2048)
    words = ws.view(torch.int64).cpu()
    at = words.nonzero().flatten()
    at = at[at >= 10 * (tiles + groups)]
    assert len(at) >= 4 * 6 * 3 * groups  # three whole tiles inside each sequence at the least
    assert set((at % 8).tolist()) == {0, 1, 2, 3, 4, 5}
