"""Evaluations of one state by the walks that several wavefronts share repeat bit for
bit: sizes on both sides of every change of the walk's shape, both laws."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("law", [0, 1])
@pytest.mark.parametrize("n,theta", [(3000, 0.6), (12289, 0.6), (24577, 0.6), (65537, 0.6), (131072, 0.6),
                                     (524288, 0.9), (524289, 0.9)])
def test_walks_repeat(gpu, n, theta, law):
    pu = gpu
    pos, vel, mass = pu.ic_plummer(n, 0x5EED0820 + n)
    cfg = pu.default_config(method=pu.METHOD_BARNES_HUT, law=law, softening=4e-4, theta=theta)
    with pu.NBodySim(cfg) as sim:
        sim.init_soa(pos, vel, mass)
        first = sim.accelerations()
        for _ in range(12):
            assert np.array_equal(sim.accelerations(), first)
