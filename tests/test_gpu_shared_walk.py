"""Walks shared by several wavefronts: both sides of every size at which the
group or the number of wavefronts changes, systems smaller than one group, and
coincident particles (buckets) in shared walks.

Interaction counts against the restated octree with FP64 centres of mass to 1e-5
and forces to 1e-5 for all but one particle in a thousand (a decision within the
rounding of a centre of mass can fall the other way); bitwise repeatable."""
import numpy as np
import pytest

from helpers import rel_err_rows

pytestmark = pytest.mark.gpu

SOFT = 4e-4


def check(pu, oracle, pos, mass, theta):
    cfg = pu.default_config(method=pu.METHOD_BARNES_HUT, law=pu.LAW_R, softening=SOFT, theta=theta)
    with pu.NBodySim(cfg) as sim:
        sim.init_soa(pos, np.zeros_like(pos), mass)
        a = sim.accelerations()
        again = sim.accelerations()
        st = sim.bh_stats()
    assert np.array_equal(a, again)
    assert st["stack_overflow"] == 0
    lo, size = oracle.dynamic_root(pos)
    F, info = oracle.bh_forces(pos, mass, theta, lo, size, G=1.0, S=SOFT, com_fp64=True)
    ref = F / mass[:, None]
    assert abs(st["interactions"] - info["interactions"]) <= 1e-5 * info["interactions"]
    assert np.count_nonzero(rel_err_rows(a, ref) >= 1e-5) <= 1e-3 * len(pos)


@pytest.mark.parametrize("n,theta", [(2, 0.6), (15, 0.6), (16, 0.6), (33, 0.6), (777, 0.4), (12288, 0.6),
                                     (12289, 0.6), (24576, 0.7), (24577, 0.7), (163840, 0.8), (163841, 0.8),
                                     (786432, 1.0), (786433, 1.0), (2621440, 1.5), (2621441, 1.5)])
def test_shapes_against_the_octree(gpu, oracle, n, theta):
    pos, _, mass = gpu.ic_plummer(n, 0x5EED0600 + n)
    check(gpu, oracle, pos, mass, theta)


@pytest.mark.parametrize("n,points", [(40, 1), (3000, 40), (20000, 7), (30000, 3000)])
def test_buckets_in_shared_walks(gpu, n, points):
    """At theta 0, buckets pair by pair included, the direct sum."""
    pu = gpu
    rng = np.random.default_rng(n)
    sites = rng.normal(size=(points, 3))
    pos = np.concatenate([sites[rng.integers(0, points, n - 1)], [[3.0, 3.0, 3.0]]]).astype(np.float32)
    mass = rng.uniform(0.5, 1.5, n) / n
    acc = []
    for method in (pu.METHOD_DIRECT, pu.METHOD_BARNES_HUT):
        with pu.NBodySim(pu.default_config(method=method, law=pu.LAW_R, softening=SOFT, theta=0.0)) as sim:
            sim.init_soa(pos, np.zeros_like(pos), mass)
            acc.append(sim.accelerations())
            if method == pu.METHOD_BARNES_HUT:
                assert sim.bh_stats()["interactions"] == n * (n - 1)
    assert rel_err_rows(acc[1], acc[0]).max() < 1e-5
