"""The sort's tiles hold 2,048 keys up to 524,288 particles and 4,096 beyond:
keys and the stable order equal the oracle's bit for bit at the edges of the
small tile and on both sides of the size at which the tile changes."""
import numpy as np
import pytest

from test_gpu_bh_sort import positions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["random", "few points"])
@pytest.mark.parametrize("n", [2047, 2048, 2049, 6145, 524288, 524289])
def test_keys_and_order_at_small_tile_edges(gpu, oracle, n, kind):
    pu = gpu
    pos = positions(kind, n)
    cfg = pu.default_config(method=pu.METHOD_BARNES_HUT, law=pu.LAW_R, softening=1e-2, theta=1.5)
    with pu.NBodySim(cfg) as sim:
        sim.init_soa(pos, np.zeros_like(pos), np.full(n, 1.0 / n))
        sim.accelerations()
        keys, order = sim.bh_tree_order()
    lo, size = oracle.dynamic_root(pos)
    ref_keys, _ = oracle.morton_keys(pos, lo, size)
    ref_order = oracle.sort_order(ref_keys)
    assert np.array_equal(order, ref_order)
    assert np.array_equal(keys, ref_keys[ref_order])
