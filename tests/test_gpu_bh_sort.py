"""The sort's tiles (4,096 keys, eight a thread) and merges (1,024 or 4,096
outputs a workgroup, the latter above 1,048,576 particles): keys and the stable
order equal the oracle's bit for bit at the edges of both, for orders in which
one run of a merge is exhausted first and for many equal keys."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def positions(kind, n):
    rng = np.random.default_rng(0x5057 + n)
    pos = rng.normal(size=(n, 3)).astype(np.float32)
    if kind == "few points":
        pos = pos[rng.integers(0, min(n, 5), n)]
    elif kind != "random":
        pos[:, 0] = np.sort(pos[:, 0]) * 1000.0  # nearly in key order
        if kind == "descending":
            pos = pos[::-1]
    return np.ascontiguousarray(pos)


@pytest.mark.parametrize("kind", ["random", "ascending", "descending", "few points"])
@pytest.mark.parametrize("n", [2, 7, 8, 9, 513, 4095, 4096, 4097, 8193, 12289, 20480, 1048576, 1048577])
def test_keys_and_order_at_tile_and_merge_edges(gpu, oracle, n, kind):
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
    if (pos == pos[0]).all():  # no extent: the cell indices exceed 64 bits, so their values are unspecified
        assert (keys == keys[0]).all()
    else:
        assert np.array_equal(keys, ref_keys[ref_order])
