"""The mass prefix of small systems in one workgroup per quantity: both sides of
the sizes at which the elements per thread change (4,096) and the chunked prefix
begins (6,144), and systems of a few particles.  Every cell's FP64 mass and
centre of mass against sums of its own particles, to the few roundings of an FP64
sum's terms (1e-12 of the mass, FP32 rounding of the centre: 1e-6 of the cell's
extent from the origin)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 17, 1000, 4095, 4096, 6143, 6144])
def test_cell_sums(gpu, n):
    pu = gpu
    pos, vel, _ = pu.ic_plummer(n, 0x5EED0900 + n)
    mass = np.random.default_rng(n).uniform(0.5, 1.5, n)
    mass[n // 2] = 0.0
    cfg = pu.default_config(method=pu.METHOD_BARNES_HUT, law=pu.LAW_R, softening=1e-2, theta=0.8)
    with pu.NBodySim(cfg) as sim:
        sim.init_soa(pos, vel, mass)
        sim.accelerations()
        _, order = sim.bh_tree_order()
        cells = sim.bh_cells()
    p, m = pos[order].astype(np.longdouble), mass[order].astype(np.longdouble)
    assert len(cells) > 0 and cells["count"].max() == n
    for c in cells:
        k = slice(int(c["first"]), int(c["first"]) + int(c["count"]))
        total = m[k].sum()
        assert abs(c["mass"] - float(total)) <= 1e-12 * float(total)
        if total > 0:
            com = (m[k, None] * p[k]).sum(axis=0) / total
            assert np.abs(c["com"] - com.astype(np.float64)).max() <= 1e-6 * max(1.0, float(np.abs(p[k]).max()))
