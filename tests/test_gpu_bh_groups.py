"""The traversal's wavefronts hold 8, 16, 32 or 64 particles by the system's
size: both sides of every size at which that changes, and systems smaller than
one wavefront.

Against the restated octree (FP64 centres of mass): the interaction count to
1e-5 relative (every particle keeps its own set of interactions whatever the
group), and forces to the repository's 1e-5 for all but the particles whose
decision at some cell lies within the rounding of its centre of mass, whose
sums the device and the octree round in different orders: a decision taken the
other way changes the count by a few, so the count's tolerance leaves room for
such particles among fewer than one in a thousand (at 98,304 the octree and the
device differ on four, whatever the group).  At theta 0 no decision is taken,
and every particle is compared with the direct sum."""
import numpy as np
import pytest

from helpers import rel_err_rows

pytestmark = pytest.mark.gpu

SOFT = 4e-4


@pytest.mark.parametrize("n,theta", [(2, 0.6), (7, 0.6), (8, 0.6), (9, 0.6), (17, 0.5), (65, 0.5), (1000, 0.3),
                                     (24576, 0.6), (24577, 0.6), (98304, 0.7), (98305, 0.7), (786432, 1.0),
                                     (786433, 1.0)])
def test_group_sizes_against_the_octree(gpu, oracle, n, theta):
    pu = gpu
    pos, vel, mass = pu.ic_plummer(n, 0x5EED0500 + n)
    cfg = pu.default_config(method=pu.METHOD_BARNES_HUT, law=pu.LAW_R, softening=SOFT, theta=theta)
    with pu.NBodySim(cfg) as sim:
        sim.init_soa(pos, vel, mass)
        a = sim.accelerations()
        again = sim.accelerations()
        st = sim.bh_stats()
    assert np.array_equal(a, again)
    lo, size = oracle.dynamic_root(pos)
    F, info = oracle.bh_forces(pos, mass, theta, lo, size, G=1.0, S=SOFT, com_fp64=True)
    ref = F / mass[:, None]
    err = rel_err_rows(a, ref)
    assert np.count_nonzero(err >= 1e-5) <= 1e-3 * n
    assert st["stack_overflow"] == 0
    assert abs(st["interactions"] - info["interactions"]) <= 1e-5 * info["interactions"]


@pytest.mark.parametrize("n", [9, 65, 5000, 24577, 98305])
def test_theta_zero_is_the_direct_sum_for_law_p(gpu, n):
    """At theta 0 every pair goes through the list: the slots' shares and the
    padding of the last round leave no pair out and add none."""
    pu = gpu
    pos, vel, mass = pu.ic_plummer(n, 0x5EED0510 + n)
    mass[n // 2] = 0.0
    acc = []
    for method in (pu.METHOD_DIRECT, pu.METHOD_BARNES_HUT):
        with pu.NBodySim(pu.default_config(method=method, law=pu.LAW_P, softening=SOFT, theta=0.0)) as sim:
            sim.init_soa(pos, vel, mass)
            acc.append(sim.accelerations())
            if method == pu.METHOD_BARNES_HUT:
                assert sim.bh_stats()["interactions"] == n * (n - 1)
    assert rel_err_rows(acc[1], acc[0]).max() < 1e-5


def test_coincident_particles_in_small_groups(gpu):
    """A bucket of identical positions is evaluated pair by pair in every group."""
    pu = gpu
    n = 300
    pos, vel, mass = pu.ic_plummer(n, 0x5EED0520)
    pos[100:161] = pos[100]
    with pu.NBodySim(pu.default_config(method=pu.METHOD_BARNES_HUT, law=pu.LAW_R, softening=SOFT, theta=0.0)) as sim:
        sim.init_soa(pos, vel, mass)
        a = sim.accelerations()
        assert sim.bh_stats()["interactions"] == n * (n - 1)
    with pu.NBodySim(pu.default_config(law=pu.LAW_R, softening=SOFT)) as sim:
        sim.init_soa(pos, vel, mass)
        want = sim.accelerations()
    assert rel_err_rows(a, want).max() < 1e-5
