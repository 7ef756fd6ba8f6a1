"""Batch systems on both sides of 1,024 particles, where the sum over unordered
pairs begins: one-sided systems drained with the pair tasks or, without any, by
their own kernel; sizes with one block and a short second one; bit for bit the
same alone and in a mix, with plain launches and graphs, and under every tuning
of the one-sided kernel; against FP64 to the repository's 1e-5 per particle."""
import numpy as np
import pytest

from helpers import rel_err_rows

pytestmark = pytest.mark.gpu

SOFT, DT = 1e-4, 1e-3
SIZES = [1, 255, 256, 257, 1000, 1024, 1025, 1280, 1281, 2047, 2049, 3000, 5000]


def _system(pu, n, seed):
    pos, vel, mass = pu.ic_plummer(max(n, 2), seed)
    pos, vel, mass = pos[:n], vel[:n], mass[:n]
    if n % 2:
        mass = mass * np.random.default_rng(seed).uniform(0.2, 2.0, n)
    return pos, vel, mass


@pytest.mark.parametrize("law", [0, 1])
def test_alone_and_together(gpu, oracle, law):
    pu = gpu
    cfg = pu.default_config(law=law, softening=SOFT)
    sets = [_system(pu, n, 0x5EED0700 + n) for n in SIZES]
    mixed = {}
    for graph in (False, True):
        for tuning in ((1, 256, 8), (2, 128, 4)):
            with pu.Batch(cfg, 30000) as b:
                b.set_graph(graph)
                b.set_tuning(*tuning)
                ids = [b.add(*s) for s in sets]
                b.step(DT, 1)
                first = [b.read(i)[2] for i in ids]
                b.step(DT, 2)
                mixed[graph, tuning] = [b.read(i) for i in ids]
    for k, (pos, vel, mass) in enumerate(sets):
        with pu.Batch(cfg, 6000) as b:
            i = b.add(pos, vel, mass)
            b.step(DT, 3)
            alone = b.read(i)
        for key, got in mixed.items():
            for x, y in zip(got[k], alone):
                assert np.array_equal(x, y), (SIZES[k], key)
        if SIZES[k] > 1:
            ref = oracle.fp64_accel(law, pos, mass, 1.0, SOFT, rows=np.arange(SIZES[k]))
            assert rel_err_rows(first[k], ref).max() < 1e-5, SIZES[k]
