"""Potential energy to the rounding of its common factors: the device's pair sums and
the host's sum of their thousands of partial sums against exactly rounded sums
(math.fsum) of FP64 pair potentials.

Bound, 5e-16 of the energy: sqrt(S), 1 / sqrt(S) and the division by it are common to
every pair (three roundings of at most 1.1e-16 each), the result one more; the pairs'
own roundings and those of the sums within a workgroup are of either sign in 1e8
terms.  The partial sums added plainly give about 0.3 x 1.1e-16 x sqrt(partials / 3) at
random and several times that where they run one way: 1.3e-15 at 20,000."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SOFT = 2.5e-3


def _potential(pos, mass, law):
    x = pos.astype(np.float64)
    rs = math.sqrt(SOFT)
    total = []
    for i in range(len(x) - 1):
        d = x[i + 1:] - x[i]
        r2 = (d * d).sum(1)
        g = np.arctan2(rs, np.sqrt(r2)) / rs if law == 0 else 1.0 / np.sqrt(r2 + SOFT)
        total.append(-mass[i] * math.fsum(mass[i + 1:] * g))
    return math.fsum(total)


@pytest.mark.parametrize("n,law", [(3000, 0), (3000, 1), (12000, 0), (12000, 1), (20000, 0)])
def test_potential_energy(gpu, n, law):
    pu = gpu
    pos, vel, mass = pu.ic_disc_bulge(n, 0x5EED0830 + n, bulge_fraction=0.2)
    with pu.NBodySim(pu.default_config(law=law, softening=SOFT)) as sim:
        sim.init_soa(pos, vel, mass)
        got = sim.diagnostics()["potential"]
    want = _potential(pos, mass, law)
    assert abs(got - want) <= 5e-16 * abs(want), (got - want) / want
