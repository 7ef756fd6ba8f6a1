"""A batch whose partial sums find no room on the device: failed allocations stand in
for a full one (nbody_config.inject_rows_failures).  What the batch already holds is
used, in more groups; systems that do not fit it alone are summed one-sided, to 1e-5
of the pairs; and the next change of the systems asks for the room again, so that the
batch's bits are those of one that was never short of it.  Also a system too large
for any rows (above about 247,000 particles): the same bits alone and in the mix."""
import numpy as np
import pytest

from helpers import rel_err_rows

pytestmark = pytest.mark.gpu

SOFT, DT = 1e-4, 1e-5


def _batch(pu, failures, capacity=100000):
    cfg = pu.default_config(law=pu.LAW_R, softening=SOFT)
    cfg.inject_rows_failures = failures
    return pu.Batch(cfg, capacity)


def _sphere(pu, n):
    return pu.ic_plummer(n, 0x5EED0840 + n)


def test_room_is_asked_for_again(gpu):
    pu = gpu
    sizes = (500, 4096, 9000)
    with _batch(pu, 1) as short, _batch(pu, 0) as free:
        ids = [short.add(*_sphere(pu, n)) for n in sizes]
        assert ids == [free.add(*_sphere(pu, n)) for n in sizes]
        for b in (short, free):
            b.step(DT, 2)
        for k, n in zip(ids, sizes):
            a, c = short.read(k), free.read(k)
            assert rel_err_rows(a[2], c[2]).max() < 1e-5
            assert np.array_equal(a[2], c[2]) == (n <= 1024)  # one-sided either way up to there
        state = {k: short.read(k) for k in ids}
        late = short.add(*_sphere(pu, 2000))
        short.step(DT, 2)
        got = {k: short.read(k) for k in ids}
        first = short.read(late)
    for k, n in zip(ids, sizes):
        with _batch(pu, 0) as b:
            i = b.add(state[k][0], state[k][1], _sphere(pu, n)[2])
            b.step(DT, 2)
            for x, y in zip(got[k], b.read(i)):
                assert np.array_equal(x, y), n
    with _batch(pu, 0) as b:
        i = b.add(*_sphere(pu, 2000))
        b.step(DT, 2)
        for x, y in zip(first, b.read(i)):
            assert np.array_equal(x, y)


def test_the_rows_held_are_used(gpu):
    pu = gpu
    later = (4096, 4097, 3000, 20000, 500)
    out = []
    for failures in (2, 0):
        with _batch(pu, failures) as b:
            ids = [b.add(*_sphere(pu, 9000))]
            b.step(DT, 1)
            ids += [b.add(*_sphere(pu, n)) for n in later]
            b.step(DT, 2)
            out.append([b.read(k) for k in ids])
    for n, a, c in zip((9000,) + later, *out):
        if n == 20000:  # does not fit the rows of 9,000
            assert rel_err_rows(a[2], c[2]).max() < 1e-5
            assert not np.array_equal(a[2], c[2])
        else:
            for x, y in zip(a, c):
                assert np.array_equal(x, y), n


def test_a_system_too_large_for_rows(gpu):
    pu = gpu
    sizes = (250000, 8000, 500)
    with _batch(pu, 0, 260000) as b:
        ids = [b.add(*_sphere(pu, n)) for n in sizes]
        b.step(DT, 1)
        mixed = [b.read(k) for k in ids]
    for n, got in zip(sizes, mixed):
        with _batch(pu, 0, 251000) as b:
            i = b.add(*_sphere(pu, n))
            b.step(DT, 1)
            for x, y in zip(got, b.read(i)):
                assert np.array_equal(x, y), n
