"""Massless particles that have no finite position (removed ones, marked by NaN; ones
that overflowed) under law R: they pull nothing, so every other particle has the
acceleration, bit for bit, that it has with them at finite places (every one of
their terms is exactly 0 either way), and their own is NaN along what is not
finite.  Through every direct sum that a size or a launch shape chooses, as single
systems and in a batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SOFT, DT = 1e-4, 1e-3
LOST = {3: (np.nan, 0.5, 0.5), 260: (np.inf, 0.5, -0.5), 517: (-np.inf, np.inf, 0.25), -1: (np.nan, np.nan, np.nan)}


def _system(pu, n, equal):
    pos, vel, mass = pu.ic_plummer(n, 0x5EED0810 + n)
    if not equal:
        mass = mass * np.random.default_rng(n).uniform(0.2, 2.0, n)
    lost = np.array(sorted(k % n for k in LOST))
    mass = mass.copy()
    mass[lost] = 0.0
    gone = pos.copy()
    for k, p in LOST.items():
        gone[k] = p
    return pos, gone, vel, mass, lost


def _check(acc, after, pos, want, lost):
    keep = np.ones(len(pos), bool)
    keep[lost] = False
    assert np.isfinite(want).all() and np.isfinite(after[keep]).all()
    assert np.array_equal(acc[keep], want[keep])
    for k in lost:
        expect = np.full(3, np.nan) if np.isnan(pos[k]).any() else np.where(np.isinf(pos[k]), np.nan, 0.0)
        assert np.array_equal(acc[k], expect, equal_nan=True), (k, acc[k])


@pytest.mark.parametrize("equal", [True, False])
@pytest.mark.parametrize("n,shape", [(1000, {}), (5000, {}), (16129, {}), (40000, {}),
                                     (5000, dict(tune_i_per_lane=1, tune_block=256))])
def test_single_systems(gpu, n, shape, equal):
    pu = gpu
    pos, gone, vel, mass, lost = _system(pu, n, equal)
    cfg = pu.default_config(law=pu.LAW_R, softening=SOFT, **shape)
    with pu.NBodySim(cfg) as sim:
        sim.init_soa(pos, vel, mass)
        want = sim.accelerations()
        sim.init_soa(gone, vel, mass)
        acc = sim.accelerations()
        sim.step(DT, 2)
        after, _, _ = sim.read_soa()
    _check(acc, after, gone, want, lost)


@pytest.mark.parametrize("n", [1000, 2000, 9000])
def test_batch(gpu, n):
    pu = gpu
    pos, gone, vel, mass, lost = _system(pu, n, False)
    with pu.Batch(pu.default_config(law=pu.LAW_R, softening=SOFT), 2 * n + 1024) as b:
        there, away = b.add(pos, vel, mass), b.add(gone, vel, mass)
        b.step(DT, 1)
        _, _, want = b.read(there)
        after, _, acc = b.read(away)
    _check(acc, after, gone, want, lost)
