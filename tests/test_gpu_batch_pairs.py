"""Batch systems that take the sum over unordered pairs: around 8,192 particles,
one and several blocks' remainders, both cuts of the
streamed blocks, equal and unequal masses, both laws; alone and in the mix bit
for bit, against FP64, and with systems joining and leaving so that groups,
tasks and the rows' buffer are laid out anew.

Tolerances: the repository's 1e-5 per particle against FP64."""
import numpy as np
import pytest

from helpers import rel_err_rows

pytestmark = pytest.mark.gpu

SOFT, DT = 1e-4, 1e-3


def _system(pu, n, equal, seed):
    pos, vel, mass = pu.ic_plummer(n, seed)
    if not equal:
        rng = np.random.default_rng(seed)
        mass = mass * rng.uniform(0.2, 2.0, n)
        mass[rng.integers(0, n, 9)] = 0.0
    return pos, vel, mass


SIZES = [(300, True), (7936, True), (7937, False), (8193, True), (9000, False), (16384, True), (16385, False),
         (30001, True)]


@pytest.mark.parametrize("law", [0, 1])
def test_mixed_sizes_alone_and_together(gpu, oracle, law):
    pu = gpu
    cfg = pu.default_config(law=law, softening=SOFT)
    sets = [_system(pu, n, eq, 0x5EED0600 + n) for n, eq in SIZES]
    with pu.Batch(cfg, 120000) as b:
        ids = [b.add(*s) for s in sets]
        b.step(DT, 1)
        first = [b.read(i)[2] for i in ids]
        b.step(DT, 2)
        mixed = [b.read(i) for i in ids]
    for k, (pos, vel, mass) in enumerate(sets):
        with pu.Batch(cfg, 40000) as b:
            i = b.add(pos, vel, mass)
            for _ in range(3):
                b.step(DT, 1)
            alone = b.read(i)
        for x, y in zip(mixed[k], alone):
            assert np.array_equal(x, y), SIZES[k]
        rows = np.unique(np.linspace(0, len(mass) - 1, 100).astype(np.int64))
        ref = oracle.fp64_accel(law, pos, mass, 1.0, SOFT, rows=rows)
        assert rel_err_rows(first[k][rows], ref).max() < 1e-5, SIZES[k]


def test_joining_and_leaving(gpu):
    pu = gpu
    cfg = pu.default_config(law=pu.LAW_R, softening=SOFT)
    a, c, d = (_system(pu, n, True, 0x5EED0610 + n) for n in (9000, 20000, 500))
    with pu.Batch(cfg, 100000) as b:
        ia = b.add(*a)
        b.step(DT, 1)
        ic = b.add(*c)       # a larger one first in the queue, a larger rows buffer
        idd = b.add(*d)
        b.step(DT, 1)
        b.remove(ia)
        b.step(DT, 1)
        ia2 = b.add(*a)
        b.step(DT, 2)
        got = {k: b.read(i) for k, i in (("a", ia2), ("c", ic), ("d", idd))}
        b.remove(ic)
        b.remove(ia2)
        b.step(DT, 1)        # one-sided systems only
        last = b.read(idd)
    for key, s, steps in (("a", a, 2), ("c", c, 4), ("d", d, 4)):
        with pu.Batch(cfg, 30000) as b:
            i = b.add(*s)
            b.step(DT, steps)
            for x, y in zip(got[key], b.read(i)):
                assert np.array_equal(x, y), key
            if key == "d":
                b.step(DT, 1)
                for x, y in zip(last, b.read(i)):
                    assert np.array_equal(x, y)


def test_plain_launches_and_device_states_match(gpu):
    """Graph off equals graph on, and a sphere generated on the device equals
    the same sphere generated by a single-system handle and added."""
    pu = gpu
    cfg = pu.default_config(law=pu.LAW_R, softening=SOFT)
    n = 12345
    with pu.NBodySim(cfg) as sim:
        sim.init_plummer(n, 77)
        pos, vel, _ = sim.read_soa()
    out = []
    for graph in (True, False):
        with pu.Batch(cfg, 40000) as b:
            b.set_graph(graph)
            i = b.add_plummer(n, 77)
            j = b.add(*_system(pu, 9000, False, 5))
            for _ in range(3):
                b.step(DT, 2)
                b.synchronize()
            out.append((b.read(i), b.read(j)))
    for x, y in zip(out[0], out[1]):
        for u, w in zip(x, y):
            assert np.array_equal(u, w)
    with pu.NBodySim(cfg) as sim:
        sim.init_soa(pos, vel, np.full(n, 1.0 / n))
        sim.step(DT, 6)
        p, _, _ = sim.read_soa()
    assert rel_err_rows(out[0][0][0], p).max() < 1e-5
