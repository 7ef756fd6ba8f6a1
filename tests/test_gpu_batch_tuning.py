"""A batch's tuning reaches the kernels that run: with pairs in the batch the
workgroups per CU are the pair kernel's, the tuner tries only them, and no tuning
changes a bit of the results."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SOFT, DT = 1e-4, 1e-6


def _filled(pu, sizes):
    b = pu.Batch(pu.default_config(law=pu.LAW_R, softening=SOFT), 200000)
    return b, [b.add_plummer(n, 0x5EED0850 + n) for n in sizes]


def _ms(b):
    t = []
    for _ in range(5):
        b.step(DT, 2)
        t.append(b.timing().step_ms)
    return sorted(t)[2]


def test_workgroups_per_cu_reach_the_pair_kernel(gpu):
    """One workgroup of four wavefronts per CU leaves a SIMD one wavefront, which waits
    for each of its own results: far from the time with six."""
    b, ids = _filled(gpu, (30000, 20000, 10000, 700))
    with b:
        b.set_tuning(1, 256, 8)
        full = _ms(b)
        b.set_tuning(1, 256, 1)
        one = _ms(b)
    assert one > 1.3 * full


def test_results_do_not_depend_on_the_tuning(gpu):
    out = []
    for wg in (1, 3, 6, 64):
        b, ids = _filled(gpu, (9000, 3000, 700))
        with b:
            b.set_tuning(2, 128, wg)
            b.step(1e-3, 3)
            out.append([b.read(k) for k in ids])
    for other in out[1:]:
        for a, c in zip(out[0], other):
            for x, y in zip(a, c):
                assert np.array_equal(x, y)


def test_the_tuner_keeps_what_it_does_not_try(gpu):
    b, ids = _filled(gpu, (9000, 3000, 700))
    with b:
        b.set_tuning(2, 128, 4)
        before = [b.read(k) for k in ids]
        t = b.tune(DT)
        assert (t["i_per_lane"], t["block"]) == (2, 128) and t["wg_per_cu"] in (2, 4, 8) and t["ms_per_step"] > 0
        for a, k in zip(before, ids):
            for x, y in zip(a[:2], b.read(k)[:2]):
                assert np.array_equal(x, y)
