"""The field of few points, whose sources are shared out over workgroups, loses nothing
between the workgroups' sums: where every term and every tile's sum is exact the
result is the exact sum rounded once.

All sources at unit distance from the points with masses that are powers of two, no
softening: law R's term is the mass itself (the reciprocal square root of a power of
four).  A tile of 256 masses of 1 to 2^-13 takes at most 22 bits, its sum is exact in
FP32; the chunks' and the whole sum take up to 31.  Bound: half an ulp, and 1/100 for
what the records of 16 chunks' sums leave out (1/1,000 of a chunk's ulp each)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(262144, 4096), (262144, 1000), (1000000, 300)])
def test_the_sum_is_rounded_once(gpu, n, m):
    pu = gpu
    worst = []
    with pu.NBodySim(pu.default_config(law=pu.LAW_R, softening=0.0)) as sim:
        for seed in range(24):
            rng = np.random.default_rng(seed)
            mass = 2.0 ** -rng.integers(0, 14, n)
            mass[0] = 1.0
            pos = np.tile(np.array([1.0, 0.0, 0.0], np.float32), (n, 1))
            sim.init_soa(pos, None, mass)
            points = np.zeros((m, 3), np.float32)
            points[1::2] = (1.0, -1.0, 0.0)
            a = sim.field(points)
            total = math.fsum(mass)
            ulp = 2.0 ** (math.floor(math.log2(total)) - 23)
            worst.append(np.abs(a[0::2, 0].astype(np.float64) - total).max() / ulp)
            worst.append(np.abs(a[1::2, 1].astype(np.float64) - total).max() / ulp)
            assert not a[0::2, 1:].any() and not a[1::2, 0].any()
    assert max(worst) <= 0.51, max(worst)
