"""Walks of four wavefronts with a list for each half of the group (bh.hip): two
wavefronts share a list, and between two barriers neither writes an entry that the
other reads or writes.  Checked on the CPU over the list's life, for all the
lengths that steps of random sizes make, with the barriers that the kernel has:

    a step's entries put at the list's end - barrier - the whole rounds beyond what
    stays evaluated by both - (the next step's first barrier, or after the last step
    the one before the padding) - the end padded by the first - barrier - the rest
    evaluated by both."""
import pathlib
import random
import re

import pytest

SRC = re.sub(r"\s+", " ", re.sub(r"//[^\n]*", "", (pathlib.Path(__file__).resolve().parents[1] /
             "procedural-universe_amd" / "csrc" / "bh.hip").read_text()))
WAVES, FLUSH, ROUND = 4, 16, 16  # wavefronts, kOwnFlush, kRound


def end_barriers():
    """Whether the kernel waits before the padding, and between it and the last evaluation."""
    tail = SRC[SRC.index("const int rest = half == 0 ? len[0] : len[1];"):]
    pad, last = tail.index("put(half, rest + lane,"), tail.index("evaluate(0, whole)")
    return "__syncthreads()" in tail[:pad], "__syncthreads()" in tail[pad:last]


def stretches(steps, before_padding, after_padding):
    """(entries read by both, entries written) between each two barriers."""
    out, length, reads, writes = [], 0, set(), set()

    def barrier():
        nonlocal reads, writes
        out.append((reads, writes))
        reads, writes = set(), set()

    for put in steps:
        barrier()
        writes |= set(range(length, length + put))
        length += put
        barrier()
        if length >= FLUSH:
            stay = length & (ROUND - 1)
            reads |= set(range(stay, length))
            length = stay
    if before_padding:
        barrier()
    whole = (length + ROUND - 1) & ~(ROUND - 1)
    writes |= set(range(length, whole))
    if after_padding:
        barrier()
    reads |= set(range(whole))
    barrier()
    return out


@pytest.mark.parametrize("seed", range(12))
def test_no_entry_is_read_while_it_is_written(seed):
    rng = random.Random(seed)
    steps = [rng.choice([1, rng.randrange(16), rng.randrange(64 * WAVES + 1)]) for _ in range(rng.randrange(1, 40))]
    for reads, writes in stretches(steps + [37], *end_barriers()):
        assert not reads & writes
