"""Walks of four or two wavefronts with a list for each half of the group: the ends
of their ranges of sizes, a last group of one particle, both laws, and coincident
particles.

Bounds as for the other shapes of the walk: interaction counts against the
restated octree with FP64 centres of mass to 1e-5, forces to 1e-5 for all but one
particle in a thousand, bitwise repeatable; at theta 0 every particle against the
direct sum, to 1e-5 of its acceleration or, where the pulls cancel, of the median
one (the rounding of either sum is about 3e-8 of that)."""
import numpy as np
import pytest

from helpers import rel_err_rows

pytestmark = pytest.mark.gpu

SOFT = 4e-4


@pytest.mark.parametrize("n,theta", [(65536, 0.6), (65537, 0.6), (200003, 0.6), (393216, 0.9), (393217, 0.9),
                                     (400003, 0.7), (524288, 0.9), (524289, 0.9), (600000, 1.0), (3000001, 2.0)])
def test_half_lists_against_the_octree(gpu, oracle, n, theta):
    pu = gpu
    pos, _, mass = pu.ic_plummer(n, 0x5EED0700 + n)
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
    assert abs(st["interactions"] - info["interactions"]) <= 1e-5 * info["interactions"]
    assert np.count_nonzero(rel_err_rows(a, F / mass[:, None]) >= 1e-5) <= 1e-3 * n


@pytest.mark.parametrize("n,points,law", [(65537, 7000, "R"), (65537, 65536, "P"), (70000, 3, "R"),
                                          (393217, 40000, "R"), (393217, 40000, "P"), (393217, 393216, "R"),
                                          (524289, 50000, "P"), (524289, 524288, "R")])
def test_half_lists_at_theta_zero(gpu, n, points, law):
    """Every pair counted; with fewer points than particles, buckets."""
    pu = gpu
    rng = np.random.default_rng(points)
    sites = rng.normal(size=(points, 3))
    which = rng.integers(0, points, n - 1) if points < n - 1 else np.arange(points)
    pos = np.concatenate([sites[which], [[3.0, 3.0, 3.0]]]).astype(np.float32)
    mass = rng.uniform(0.5, 1.5, n) / n
    acc = []
    for method in (pu.METHOD_DIRECT, pu.METHOD_BARNES_HUT):
        cfg = pu.default_config(method=method, law=pu.LAW_R if law == "R" else pu.LAW_P, softening=SOFT, theta=0.0)
        with pu.NBodySim(cfg) as sim:
            sim.init_soa(pos, np.zeros_like(pos), mass)
            acc.append(sim.accelerations().astype(np.float64))
            if method == pu.METHOD_BARNES_HUT:
                assert sim.bh_stats()["interactions"] == n * (n - 1)
    size = np.linalg.norm(acc[0], axis=1)
    err = np.linalg.norm(acc[1] - acc[0], axis=1)
    assert (err / np.maximum(size, np.median(size))).max() < 1e-5
