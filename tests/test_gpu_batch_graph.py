"""A batch's captured graph after its systems changed: whichever call lays the
items out anew (the step itself, `info`, `step_sequential`), the next step with
the same (dt, nsteps) must not replay a graph of the old layout.  Systems on both
sides of 1,024 particles join and leave, so that the kinds of kernels, the number
of groups and the buffers change in both directions.  Bit for bit a fresh batch's
steps from the same state."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SOFT, DT = 1e-4, 1e-3
SMALL, LARGE = 500, 4096


def _lay_out(b, how, nsteps):
    """Have the items rebuilt before the next step; the steps this takes by itself."""
    if how == "info":
        b.info()
        return 0
    if how == "sequential":
        b.step_sequential(DT, nsteps)
        return nsteps
    return 0


def _fresh(pu, cfg, state, steps):
    with pu.Batch(cfg, 20000) as b:
        i = b.add(*state)
        b.set_graph(False)
        b.step(DT, steps)
        return b.read(i)


@pytest.mark.parametrize("how", ["info", "sequential", "step"])
@pytest.mark.parametrize("first,then", [((SMALL,), (SMALL, LARGE)), ((SMALL, LARGE), (SMALL,)), ((LARGE,), (SMALL,)),
                                        ((LARGE,), (LARGE, 9000)), ((SMALL, LARGE), (LARGE, 20000)),
                                        ((LARGE, 9000), (1000,))])
def test_a_changed_batch_takes_no_old_graph(gpu, how, first, then):
    pu = gpu
    cfg = pu.default_config(law=pu.LAW_R, softening=SOFT)
    nsteps = 2
    sets = {n: pu.ic_plummer(n, 0x5EED0800 + n) for n in {*first, *then}}
    with pu.Batch(cfg, 60000) as b:
        ids = {n: b.add(*sets[n]) for n in first}
        taken = dict.fromkeys(first, 0)
        for _ in range(2):  # captured, then replayed
            b.step(DT, nsteps)
        for n in taken:
            taken[n] += 2 * nsteps
        for n in first:
            if n not in then:
                b.remove(ids.pop(n))
        for n in then:
            if n not in ids:
                ids[n] = b.add(*sets[n])
                taken[n] = 0
        more = _lay_out(b, how, nsteps)
        for _ in range(3):  # with reads between the replays
            b.step(DT, nsteps)
            more += nsteps
            got = {n: b.read(ids[n]) for n in then}
            for n in then:
                for x, y in zip(got[n], _fresh(pu, cfg, sets[n], taken[n] + more)):
                    assert np.array_equal(x, y), (n, more)


def test_a_layout_that_returns(gpu):
    """Back to the first systems, in the buffers as they grew meanwhile."""
    pu = gpu
    cfg = pu.default_config(law=pu.LAW_R, softening=SOFT)
    a, c = pu.ic_plummer(SMALL, 0x5EED0801), pu.ic_plummer(LARGE, 0x5EED0802)
    with pu.Batch(cfg, 20000) as b:
        ia, ic = b.add(*a), b.add(*c)
        b.step(DT, 2)
        b.remove(ic)
        b.step(DT, 2)
        ic = b.add(*c)
        b.info()
        b.step(DT, 2)
        got = b.read(ia), b.read(ic)
    for state, steps, g in ((a, 6, got[0]), (c, 2, got[1])):
        for x, y in zip(g, _fresh(pu, cfg, state, steps)):
            assert np.array_equal(x, y)
