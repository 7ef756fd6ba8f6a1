"""The walk of one wavefront to a group of 64 (from 1,572,865 particles on at theta above
1.1, from 8,388,609 on at any) against the walk of two on the same decisions.

* Around theta = 1.1 both walks decide alike: the largest floats below 1.1 and
  below 1.1 + 1e-10 are the same, so the interaction counts are equal and the
  accelerations differ by the order of their sums: 1e-5, the repository's bound for
  two FP32 sums of the same terms.  With coincident particles, whose buckets each
  walk expands in its own way, and both laws.
* Around 8,388,608 particles: one more particle, without mass, changes the tree
  beside it and no force, but for particles that decide at a cell whose centre of
  mass is rounded the other way (fewer than one in a thousand, as against the
  octree)."""
import numpy as np
import pytest

from helpers import rel_err_rows

pytestmark = pytest.mark.gpu

SOFT = 4e-4


def _evaluate(pu, pos, mass, law, theta):
    cfg = pu.default_config(method=pu.METHOD_BARNES_HUT, law=law, softening=SOFT, theta=theta)
    with pu.NBodySim(cfg) as sim:
        sim.init_soa(pos, np.zeros_like(pos), mass)
        a = sim.accelerations()
        assert np.array_equal(a, sim.accelerations())
        return a, sim.bh_stats()


@pytest.mark.parametrize("n,law,sites", [(1572865, 0, 0), (1572865, 1, 0), (1600000, 0, 60000), (1600000, 1, 200),
                                         (3000001, 0, 1000000)])
def test_one_and_two_wavefronts_decide_alike(gpu, n, law, sites):
    pu = gpu
    pos, _, mass = pu.ic_plummer(n, 0x5EED0860 + n)
    if sites:
        rng = np.random.default_rng(sites)
        pos = pos[rng.integers(0, sites, n)]
        pos[:n // 2] = pu.ic_plummer(n // 2, 0x5EED0861 + n)[0]  # half of them apart
    two, st2 = _evaluate(pu, pos, mass, law, 1.1)
    one, st1 = _evaluate(pu, pos, mass, law, 1.1 + 1e-10)
    assert float(np.float32(1.1)) > 1.1 + 1e-10  # the same floats lie below both
    assert st1["stack_overflow"] == st2["stack_overflow"] == 0
    assert st1["interactions"] == st2["interactions"]
    size = np.linalg.norm(two.astype(np.float64), axis=1)
    err = np.linalg.norm(one.astype(np.float64) - two, axis=1)
    assert (err / np.maximum(size, np.median(size))).max() < 1e-5


def test_both_sides_of_the_largest_size(gpu):
    pu = gpu
    n = 8388608
    pos, _, mass = pu.ic_plummer(n, 0x5EED0862)
    two, st2 = _evaluate(pu, pos, mass, 0, 1.0)
    more = np.concatenate([pos, [[0.25, -0.5, 0.75]]]).astype(np.float32)
    one, st1 = _evaluate(pu, more, np.append(mass, 0.0), 0, 1.0)
    assert st1["stack_overflow"] == st2["stack_overflow"] == 0
    assert abs(st1["interactions"] - st2["interactions"]) <= 1e-5 * st2["interactions"]
    assert np.count_nonzero(rel_err_rows(one[:n], two) >= 1e-5) <= 1e-3 * n
