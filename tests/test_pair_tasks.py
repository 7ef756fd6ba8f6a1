"""The sum over unordered pairs covers every ordered pair of particles exactly
once, and the reduction reads exactly the rows that were written, for every plan
that single systems and batches choose, checked on the CPU.

`sym_force_kernel` (csrc/direct_sym.hip) and `batch_sym_kernel` (csrc/batch.hip)
run tasks (A, d, h): block A as residents, run h of block A + d as the stream, both
directions for d > 0, one for d = 0.  A task writes its residents' sums to one
row of partial sums and its stream's to another; `sum_rows` (direct_sym_core.hpp)
adds a particle's rows.  The formulas are read from the sources as text, so that
a change there has to come back here."""
import pathlib
import re

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "procedural-universe_amd" / "csrc"


def text(name):
    return re.sub(r"\s+", " ", (CSRC / name).read_text())


def test_the_formulas_are_the_ones_checked():
    sym, core, batch = text("direct_sym.hip"), text("direct_sym_core.hpp"), text("batch.hip")
    for part in ("if (n_pad < 16384) return p;", "p.block = ((n_pad + 191) / 192 + kStep - 1) / kStep * kStep;",
                 "p.split = tasks >= 4096 ? 1 : tasks >= 2048 ? 2 : 4;", "if (2 * d == P.nsb && a >= d) return;",
                 "core::sym_task<LAW, false, EQ>(A, S, a, a, h, h, 0);",
                 "core::sym_task<LAW, true, EQ>(A, S, a, b, h, d * P.split + h, (H + 1) * P.split + d - 1);",
                 "const dim3 grid(P.nsb, (P.nsb / 2 + 1) * P.split);"):
        assert part in sym, part
    for part in ("const int B = A.plan.block, S0 = B / A.plan.split;",
                 "const int i0 = blockA * B, i1 = min(i0 + B, A.n_pad);",
                 "const int j0 = blockB * B + h * S0, j1 = min(j0 + S0, A.n_pad);",
                 "const int H = P.nsb / 2, rows = (H + 1) * P.split + H, per = (rows + 3) / 4;",
                 "const int d = resident ? r / P.split : r - (H + 1) * P.split + 1;",
                 "if (2 * d == P.nsb && (b >= d) == resident) continue;"):
        assert part in core, part
    for part in ("p.block = 1024;", "p.split = p.nsb <= 16 ? 4 : 2;", "constexpr size_t kSymMin = 1280;",
                 "for (int a = 0; a < (d > 0 && 2 * d == P.nsb ? d : P.nsb); ++a)",
                 "const int rowi = w.d * D.sym.split + w.h, rowj = (H + 1) * D.sym.split + w.d - 1;"):
        assert part in batch, part


def single_plan(n_pad):
    block = ((n_pad + 191) // 192 + 1023) // 1024 * 1024
    nsb = -(-n_pad // block)
    tasks = nsb * (nsb + 1) // 2
    return block, nsb, 1 if tasks >= 4096 else 2 if tasks >= 2048 else 4


def batch_plan(n_pad):
    nsb = -(-n_pad // 1024)
    return 1024, nsb, 4 if nsb <= 16 else 2


def check(n_pad, block, nsb, split):
    H = nsb // 2
    run = block // split
    assert block % split == 0 and run % 256 == 0 and (nsb - 1) * block < n_pad <= nsb * block
    # ordered (target block, source block, run of the side that streams, target side)
    covered = {}
    written = {}

    def write(row, b, lo, hi):
        if lo < hi:
            for other in written.setdefault((row, b), []):
                assert hi <= other[0] or other[1] <= lo, "two tasks write the same sums"
            written[row, b].append((lo, hi))

    for a in range(nsb):
        for d in range(H + 1):
            if d > 0 and 2 * d == nsb and a >= d:
                continue
            b = (a + d) % nsb
            ra, rb = (a * block, min((a + 1) * block, n_pad)), b * block
            for h in range(split):
                j0, j1 = rb + h * run, min(rb + (h + 1) * run, n_pad)
                write(d * split + h, a, *ra)
                if j0 >= j1:
                    continue
                covered[a, b, h] = covered.get((a, b, h), 0) + 1  # targets a from run h of b
                if d > 0:
                    covered[b, a, ("stream", h)] = covered.get((b, a, ("stream", h)), 0) + 1
                    write((H + 1) * split + d - 1, b, j0, j1)
    # every ordered pair of blocks: as residents over every run, or as the stream in every run
    for t in range(nsb):
        for s in range(nsb):
            runs_s = [h for h in range(split) if s * block + h * run < n_pad]
            runs_t = [h for h in range(split) if t * block + h * run < n_pad]
            resident = [covered.get((t, s, h), 0) for h in runs_s]
            stream = [covered.get((t, s, ("stream", h)), 0) for h in runs_t]
            assert (all(v == 1 for v in resident) and not any(stream)) or \
                   (all(v == 1 for v in stream) and not any(resident)), (t, s)
    # the reduction's rows of each block are the written ones, each over the whole block
    for b in range(nsb):
        read = set()
        for r in range((H + 1) * split + H):
            resident = r < (H + 1) * split
            d = r // split if resident else r - (H + 1) * split + 1
            if 2 * d == nsb and (b >= d) == resident:
                continue
            read.add(r)
        end = min((b + 1) * block, n_pad)
        for r in read:
            pieces = sorted(written[r, b])
            assert pieces[0][0] == b * block and pieces[-1][1] == end
            assert all(x[1] == y[0] for x, y in zip(pieces, pieces[1:]))
        assert read == {r for (r, blk) in written if blk == b}


@pytest.mark.parametrize("n_pad", [16384, 16640, 17408, 20224, 24576, 32768, 33024, 65536, 65792, 100096, 131072,
                                   196608, 196864, 262144, 400128])
def test_single_system_plans(n_pad):
    check(n_pad, *single_plan(n_pad))


@pytest.mark.parametrize("n_pad", [1280, 1536, 2048, 2304, 3072, 3328, 4096, 8192, 9216, 16384, 16640, 17408, 32768,
                                   65536, 66048])
def test_batch_plans(n_pad):
    check(n_pad, *batch_plan(n_pad))
