"""Direct sums below 16,384 padded particles take a step in one launch: one and
two particles, the edges of the 8- and 16-target workgroups, of the 1,024-source
tiles and of the size where the workgroups' targets change, both laws, masses
with zeros, coincident particles; against FP64 (1e-5 per particle, 1e-6 RMS: the
repository's tolerances) and, stepped, against the one-sided kernel."""
import numpy as np
import pytest

from helpers import rel_err_rows

pytestmark = pytest.mark.gpu

SOFT = 1e-4


@pytest.mark.parametrize("law", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 7, 9, 63, 255, 1023, 1025, 2048, 2049, 3000, 4097, 12345, 16128])
def test_small_steps(gpu, oracle, n, law):
    pu = gpu
    pos, vel, mass = pu.ic_plummer(n, 0x5EED0700 + n)
    if n > 4:
        mass = mass * np.random.default_rng(n).uniform(0.2, 2.0, n)
        mass[n // 2] = 0.0
        pos[1] = pos[n - 1]
    with pu.NBodySim(pu.default_config(law=law, softening=SOFT)) as sim:
        sim.init_soa(pos, vel, mass)
        a = sim.accelerations()
        again = sim.accelerations()
        sim.step(1e-3, 3)
        p, v, _ = sim.read_soa()
    assert np.array_equal(a, again)
    if n == 1:
        assert np.all(a == 0)
    else:
        err = rel_err_rows(a, oracle.fp64_accel(law, pos, mass, 1.0, SOFT))
        assert err.max() < 1e-5 and np.sqrt(np.mean(err ** 2)) < 1e-6
    with pu.NBodySim(pu.default_config(law=law, softening=SOFT, tune_i_per_lane=1, tune_block=256, tune_split=1)) as sim:
        sim.init_soa(pos, vel, mass)
        sim.step(1e-3, 3)
        p1, v1, _ = sim.read_soa()
    scale = np.abs(p1).max()
    assert np.abs(p - p1).max() <= 1e-5 * scale and np.abs(v - v1).max() <= 1e-5 * np.abs(v1).max()
