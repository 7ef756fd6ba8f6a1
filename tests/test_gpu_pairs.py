"""The direct sum over unordered pairs (from 16,384 padded particles on): the
first size it serves and the last it does not, ragged last blocks, even and odd
numbers of blocks, every number of runs a block's stream is cut into, and
blocks of more than 1,024 particles, with equal and unequal masses (the equal
ones take a kernel of their own), massless and coincident particles, against
the FP64 sum and the one-sided kernel.

Tolerances: the repository's, accelerations to 1e-5 of FP64 per particle and
1e-6 RMS (FP32 pair terms of a few ulp in FP32 sums of 256).
"""
import numpy as np
import pytest

from helpers import rel_err_rows

pytestmark = pytest.mark.gpu

SOFT = 1e-4


def _fp64(points, pos, mass, law):
    out = np.empty((len(points), 3))
    x, m = pos.astype(np.float64), mass.astype(np.float64)
    step = max(1, (1 << 22) // len(x))
    for i in range(0, len(points), step):
        d = x[None] - points[i:i + step, None].astype(np.float64)
        r2 = (d * d).sum(-1)
        with np.errstate(divide="ignore", invalid="ignore"):
            f = np.where(r2 > 0, m / (np.sqrt(r2) * (r2 + SOFT)), 0.0) if law == 0 else m * (r2 + SOFT) ** -1.5
        out[i:i + step] = (d * f[..., None]).sum(1)
    return out


@pytest.mark.parametrize("law,equal", [(0, True), (0, False), (1, True), (1, False)])
@pytest.mark.parametrize("n", [16128, 16129, 17000, 17408, 19457, 65537, 93000, 200003])
def test_pairs_against_fp64(gpu, n, law, equal):
    pu = gpu
    pos, vel, mass = pu.ic_plummer(n, 0x5EED0400 + n)
    rng = np.random.default_rng(n)
    pos[5] = pos[n - 1]  # coincident, in different blocks
    if not equal:
        mass = mass * rng.uniform(0.1, 2.0, n)
        mass[rng.integers(0, n, 50)] = 0.0
    rows = np.unique(np.concatenate([[0, 5, 255, 256, 1023, 1024, n - 257, n - 1], rng.integers(0, n, 200)]))
    ref = _fp64(pos[rows], pos, mass, law)
    with pu.NBodySim(pu.default_config(law=law, softening=SOFT)) as sim:
        sim.init_soa(pos, vel, mass)
        a = sim.accelerations()
        again = sim.accelerations()
        sim.step(1e-3, 2)
        p, v, _ = sim.read_soa()
    assert np.array_equal(a, again)
    err = rel_err_rows(a[rows], ref)
    assert err.max() < 1e-5 and np.sqrt(np.mean(err ** 2)) < 1e-6
    with pu.NBodySim(pu.default_config(law=law, softening=SOFT, tune_i_per_lane=1, tune_block=256)) as sim:
        sim.init_soa(pos, vel, mass)
        one = sim.accelerations()
        sim.step(1e-3, 2)
        p1, v1, _ = sim.read_soa()
    assert rel_err_rows(a, one).max() < 1e-5
    assert rel_err_rows(p, p1).max() < 1e-5


def test_pairs_graph_replay_equals_plain_launches(gpu):
    pu = gpu
    n = 20011
    pos, vel, mass = pu.ic_plummer(n, 0x5EED0410)
    cfg = pu.default_config(law=pu.LAW_R, softening=SOFT)
    with pu.NBodySim(cfg) as plain, pu.NBodySim(cfg) as graph:
        graph.set_graph(True)
        for s in (plain, graph):
            s.init_soa(pos, vel, mass)
        for _ in range(4):
            for s in (plain, graph):
                s.step(1e-3, 3)
            plain.accelerations()  # eager work between the replays
            graph.accelerations()
            for x, y in zip(plain.read_soa(), graph.read_soa()):
                assert np.array_equal(x, y)


def test_a_larger_then_a_smaller_state_in_one_handle(gpu):
    """The partial sums' buffer is kept; each state's result is its own."""
    pu = gpu
    cfg = pu.default_config(law=pu.LAW_R, softening=SOFT)
    sets = [pu.ic_plummer(n, 0x5EED0420 + n) for n in (40000, 3000, 17000)]
    want = []
    for pos, vel, mass in sets:
        with pu.NBodySim(cfg) as sim:
            sim.init_soa(pos, vel, mass)
            want.append(sim.accelerations())
    with pu.NBodySim(cfg) as sim:
        for (pos, vel, mass), w in zip(sets, want):
            sim.init_soa(pos, vel, mass)
            assert np.array_equal(sim.accelerations(), w)
