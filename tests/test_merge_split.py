"""The wave-wide search for a merge's split, and the pairing of runs by the merge
launches, checked on the CPU against a stable sort: runs with ties, empty and
short runs, and every output position at which a workgroup can start."""
import pathlib
import re

import numpy as np
import pytest

SRC = re.sub(r"\s+", " ", (pathlib.Path(__file__).resolve().parents[1] / "procedural-universe_amd" / "csrc" /
                          "bh.hip").read_text())


def test_the_steps_are_the_ones_checked():
    for part in ("int lo = max(0, d - lb), hi = min(d, la);", "const int step = (hi - lo + 63) / 64;",
                 "const bool in = p < hi && A[p] <= B[d - 1 - p];", "if (step == 1) return lo + k;",
                 "if (k == 0) return lo;", "lo += (k - 1) * step + 1;", "hi = min(hi, lo + step - 1);",
                 "const int pair = o0 / (2 * run) * (2 * run);", "const int la = min(run, n - pair);",
                 "const int lb = max(0, min(run, n - pair - run));",
                 "const int from = pair + (i < na ? a0 + i : la + b0 + (i - na));",
                 "for (int run = TILE; run < n; run *= 2)"):
        assert part in SRC, part


def split(A, B, d):
    la, lb = len(A), len(B)
    lo, hi = max(0, d - lb), min(d, la)
    while lo < hi:
        step = (hi - lo + 63) // 64
        probes = [lo + lane * step for lane in range(64)]
        k = sum(1 for p in probes if p < hi and A[p] <= B[d - 1 - p])
        if step == 1:
            return lo + k
        if k == 0:
            return lo
        lo += (k - 1) * step + 1
        hi = min(hi, lo + step - 1)
    return lo


@pytest.mark.parametrize("values", [2, 10, 1 << 40])
@pytest.mark.parametrize("la,lb", [(0, 7), (7, 0), (1, 1), (63, 64), (64, 65), (200, 1000), (1000, 130), (4096, 4096)])
def test_split_is_the_stable_merge(values, la, lb):
    rng = np.random.default_rng(la * 7919 + lb)
    A, B = np.sort(rng.integers(0, values, la)), np.sort(rng.integers(0, values, lb))
    from_a = np.argsort(np.concatenate([A, B]), kind="stable") < la
    before = np.concatenate([[0], np.cumsum(from_a)])
    for d in sorted({0, 1, la + lb} | set(range(0, la + lb, 61)) | set(range(0, la + lb, 1024))):
        if d <= la + lb:
            assert split(A, B, d) == before[d], d


@pytest.mark.parametrize("tile,out", [(64, 32), (64, 128), (32, 64)])
@pytest.mark.parametrize("n", [1, 33, 64, 65, 200, 257, 511, 1024])
def test_launches_sort_stably(n, tile, out):
    """Tiles and merges as the launches take them, scaled down."""
    keys = np.random.default_rng(n).integers(0, 9, n)
    idx = np.arange(n)
    for t in range(0, n, tile):
        o = np.argsort(keys[t:t + tile], kind="stable")
        keys[t:t + tile], idx[t:t + tile] = keys[t:t + tile][o], idx[t:t + tile][o]
    run = tile
    while run < n:
        nk, ni = keys.copy(), idx.copy()
        for o0 in range(0, n, out):
            pair = o0 // (2 * run) * (2 * run)
            la, lb = min(run, n - pair), max(0, min(run, n - pair - run))
            A, B = keys[pair:pair + la], keys[pair + la:pair + la + lb]
            d0, d1 = o0 - pair, min(o0 - pair + out, la + lb)
            a0, a1 = split(A, B, d0), split(A, B, d1)
            src = np.concatenate([np.arange(pair + a0, pair + a1), np.arange(pair + la + d0 - a0, pair + la + d1 - a1)])
            o = np.argsort(keys[src], kind="stable")
            nk[o0:o0 + d1 - d0], ni[o0:o0 + d1 - d0] = keys[src][o], idx[src][o]
        keys, idx, run = nk, ni, run * 2
    want = np.argsort(np.random.default_rng(n).integers(0, 9, n), kind="stable")
    assert np.array_equal(idx, want)
