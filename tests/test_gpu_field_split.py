"""The field at few points splits the sources over workgroups and wavefronts:
every size where the split changes shape (one point, the edges of the 64-point
workgroups, one source tile, chunks that do not divide the tiles, both sides of
the 262,144 points from which the sources are not split) against the FP64 sum.

Tolerance: FP32 pair terms (a few ulp, 6e-8 each) with compensated sums of
FP32 tile sums: 1e-5 of the row, the repository's acceleration tolerance.
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


@pytest.mark.parametrize("law", [0, 1])
@pytest.mark.parametrize("n,m", [(1, 1), (255, 64), (300, 65), (257, 63), (70001, 1), (70001, 129), (33000, 2048),
                                 (300, 65537), (300, 262143), (300, 262144)])
def test_field_split_edges(gpu, n, m, law):
    pu = gpu
    pos, vel, mass = pu.ic_plummer(n, 0x5EED0310 + n)
    rng = np.random.default_rng(n + m)
    pts = rng.normal(0.0, 1.5, (m, 3)).astype(np.float32)
    pts[: m // 3] = pos[rng.integers(0, n, m // 3)]  # points on particles
    with pu.NBodySim(pu.default_config(law=law, softening=SOFT)) as sim:
        sim.init_soa(pos, vel, mass)
        got = sim.field(pts)
        again = sim.field(pts)
    assert np.array_equal(got, again)
    rows = np.unique(np.concatenate([np.arange(min(m, 300)), rng.integers(0, m, 300), [m - 1]]))
    ref = _fp64(pts[rows], pos, mass, law)
    alone = np.linalg.norm(ref, axis=1) == 0  # the only particle's own position
    assert np.all(got[rows][alone] == 0)
    assert rel_err_rows(got[rows][~alone], ref[~alone]).max(initial=0.0) < 1e-5
