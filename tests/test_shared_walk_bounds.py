"""The stack and list of a walk that several wavefronts share never overflow,
checked on the CPU.

With W wavefronts a step takes up to 8 W cells from the top of the one stack,

    all_k = min(8 W, sp, max((kCap - kDfsReserve - sp) / 7, 1)),

and pushes their opened children in their place: a batch of more than one cell
leaves the stack at most kCap - kDfsReserve high, above which cells are taken one
at a time, depth first, so the argument for a single wavefront's stack holds with
kCap in place of its capacity.  Buckets within a batch are expanded into the
lists and push nothing.

Wavefront w takes the cells w, w + W, ... of the batch, at most eight, each with at
most eight list entries, after a flush if they might not fit."""
import re

import pytest

from test_walk_bounds import BUCKET, SRC, adversarial_roots, children, kernel_constants, list_guards


def stack_cap(waves):
    src = SRC.read_text()
    body = re.search(r"constexpr int stack_cap\(int waves\) \{ return ([^;]+); \}", src).group(1)
    m = re.fullmatch(r"waves == 1 \? kStackCap : 56 \* waves \+ (\d+) \+ kDfsReserve", body)
    assert m, body
    cap, reserve, _, _ = kernel_constants()
    return cap if waves == 1 else 56 * waves + int(m.group(1)) + reserve


def shapes():
    """(group, waves) of every traversal the host chooses."""
    src = SRC.read_text()
    body = src[src.index("inline TravShape trav_shape"):]
    body = body[:body.index("\n}\n")]
    return sorted({(int(g), int(w)) for g, w in re.findall(r"return \{(\d+), (\d+)\};", body)})


def test_rules_in_the_kernel_are_the_ones_checked():
    src = re.sub(r"\s+", "", SRC.read_text())
    assert "all_k=min(min(8*W,sp),max((kCap-kDfsReserve-sp)/7,1));" in src
    assert "constintshare=W*grp+wave;" in src
    assert "k=(all_k-wave+W-1)/W;" in src
    assert "if(cnt>kListCap-8*k)flush();" in src
    assert all(w in (1, 2, 4, 8) and g in (16, 32, 64) for g, w in shapes())
    assert any(w > 1 for _, w in shapes())


@pytest.mark.parametrize("waves", [2, 4, 8])
@pytest.mark.parametrize("root", list(adversarial_roots(21)), ids=lambda r: f"full{r[2][0]}_slot{r[2][2]}")
def test_shared_walk_stays_under_the_bound(root, waves):
    _, reserve, levels, _ = kernel_constants()
    cap = stack_cap(waves)
    stack, peak = [root], 1
    while stack:
        sp = len(stack)
        k = min(8 * waves, sp, max((cap - reserve - sp) // 7, 1))
        batch = stack[-k:][::-1]
        del stack[sp - k:]
        pushed = []
        for w in range(waves):  # the first wavefront's children end on top
            for cell in batch[w::waves]:
                pushed.extend(children(cell, levels) if cell[1] != BUCKET else [])
        stack.extend(reversed(pushed))
        peak = max(peak, len(stack))
        assert peak <= cap
    assert peak <= max(cap - reserve, cap - reserve + 7 * levels)


@pytest.mark.parametrize("waves", [2, 4, 8])
def test_shares_cover_the_batch_and_fit_the_list(waves):
    cap, bucket_margin, _ = list_guards()
    for all_k in range(1, 8 * waves + 1):
        taken = []
        for w in range(waves):
            k = (all_k - w + waves - 1) // waves
            mine = [waves * g + w for g in range(8) if waves * g + w < all_k]
            assert len(mine) == k <= 8
            taken += mine
            for cnt in range(cap + 1):
                c = 0 if cnt > cap - 8 * k else cnt
                assert c + 8 * k <= cap
        assert sorted(taken) == list(range(all_k))
    assert all((0 if c > cap - bucket_margin else c) + 1 <= cap for c in range(cap + 1))
