"""The two normalising kernels hand a row or segment whose bounded wait has run out from block to block by a note
(leave_note in csrc/gae_norm.hip). Its leaver stores the note and then looks at the sums' flags; whoever publishes stores a
flag and then looks at notes. On both sides the store has to be performed before the load is served, which no result
of a run shows: the window is a few hundred nanoseconds behind a wait that ran out. So this reads the assembly that the
compiler makes of the source."""

import re
import subprocess

import pytest

from areal_amd import build

KERNELS = ("adv_gae_kernel", "gae_tile_norm_kernel")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{name: instructions} of the kernels that leave notes."""
    try:
        hipcc = build._hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    asm = tmp_path_factory.mktemp("asm") / "gae_norm.s"
    cmd = [hipcc, *build.HIPCC_FLAGS, "-ffp-contract=off", "--cuda-device-only", "-S", str(build.CSRC / "gae_norm.hip"), "-o", str(asm)]
    subprocess.run(cmd, check=True, capture_output=True)
    found = {}
    for m in re.finditer(r"^(_Z\S+):[^\n]*\n(.*?)^\.Lfunc_end", asm.read_text(), re.S | re.M):
        lines = [line.strip() for line in m.group(2).split("\n")]
        if any(k in m.group(1) for k in KERNELS) and any(line.startswith("global_atomic_cmpswap_x2") for line in lines):
            found[m.group(1)] = lines
    assert len(found) >= 8  # two forms of three estimators, with and without a lambda per sequence
    return found


def _waits(line):
    return re.match(r"s_waitcnt\b.*\bvmcnt\(0\)", line) is not None


def test_a_note_is_out_before_the_sums_are_looked_at(kernels):
    for name, lines in kernels.items():
        swaps = [i for i, line in enumerate(lines) if line.startswith("global_atomic_swap_x2")]
        assert swaps, name
        for i in swaps:
            behind = lines[i + 1 :]
            load = next(k for k, line in enumerate(behind) if re.match(r"(global|flat|buffer)_load", line))
            assert any(_waits(line) for line in behind[:load]), (name, behind[: load + 1])


def test_a_flag_is_out_before_notes_are_looked_at(kernels):
    """Each place that takes notes (by compare and swap) reads them behind a wait for everything stored before; between the
    two lie only the loads of the notes."""
    for name, lines in kernels.items():
        looks = [i for i, line in enumerate(lines) if _waits(line) and "flag out before notes are read" in line]
        takes = sum(line.startswith("global_atomic_cmpswap_x2") for line in lines)
        assert len(looks) >= takes, (name, len(looks), takes)
        for i in looks:
            behind = lines[i + 1 :]
            first = next(k for k, line in enumerate(behind) if re.match(r"(global|flat|buffer)_(load|store|atomic)", line))
            assert re.match(r"global_load_dwordx2\b.*\bsc1\b", behind[first]), (name, behind[first])


def test_a_tile_waits_once(kernels):
    """gae_tile_norm_kernel waits for maps and then for sums: both until one time. The clock is read to set it, in front of all
    else, and where the loops look at it: the two that wait, and the one that looks at sums once."""
    for name, lines in kernels.items():
        if "gae_tile_norm_kernel" not in name:
            continue
        reads = [i for i, line in enumerate(lines) if line.startswith("s_memrealtime")]
        waits = [i for i, line in enumerate(lines) if line.startswith("s_sleep")]
        assert len(reads) == 1 + 3 and len(waits) == 2, (name, reads, waits)
        for i in reads[1:]:
            assert not any(line.startswith("s_add_u32") for line in lines[i + 1 : i + 9]), (name, lines[i : i + 9])
