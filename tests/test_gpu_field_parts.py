"""The field's workgroups take a chunk's source tiles in two halves: chunks of
one tile, of an odd number and of two, and the sum of one, a few and many chunks
for point counts around the 16 of its workgroups, against the FP64 sum to the
repository's 1e-5."""
import numpy as np
import pytest

from helpers import rel_err_rows
from test_gpu_field_split import SOFT, _fp64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("law", [0, 1])
@pytest.mark.parametrize("n,m", [(256, 1), (512, 5), (768, 17), (1281, 16), (4097, 15), (20000, 33), (20000, 4097),
                                 (3000, 20000), (769, 66000)])
def test_halves_and_sums(gpu, n, m, law):
    pu = gpu
    pos, _, mass = pu.ic_plummer(n, 0x5EED0800 + n)
    pts = np.random.default_rng(n + m).normal(0.0, 1.5, (m, 3)).astype(np.float32)
    with pu.NBodySim(pu.default_config(law=law, softening=SOFT)) as sim:
        sim.init_soa(pos, np.zeros_like(pos), mass)
        got = sim.field(pts)
        again = sim.field(pts)
    assert np.array_equal(got, again)
    rows = np.unique(np.linspace(0, m - 1, 300).astype(np.int64))
    assert rel_err_rows(got[rows], _fp64(pts[rows], pos, mass, law)).max() < 1e-5
