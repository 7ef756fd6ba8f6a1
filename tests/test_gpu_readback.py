"""Reads pack the fields on the device: through pinned memory up to 8 MiB, by
way of a device buffer above, in the same handle as its size grows and shrinks.
Every size at the edges of the packing kernel's 256 records and of the 8 MiB
(three fields of 233,016 and 233,017 particles, one of 699,050 and 699,051)
against the state that was put in, exactly."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _state(n, seed):
    rng = np.random.default_rng([n, seed])
    return (rng.normal(size=(n, 3)).astype(np.float32), rng.normal(size=(n, 3)).astype(np.float32),
            rng.uniform(0.5, 2.0, n))


def test_every_size_in_one_handle(gpu):
    pu = gpu
    fp = ctypes.POINTER(ctypes.c_float)
    with pu.NBodySim(pu.default_config()) as sim:
        for n in (1, 255, 256, 257, 1000, 233016, 233017, 5000, 699050, 699051, 513):
            pos, vel, mass = _state(n, 1)
            sim.init_soa(pos, vel, mass)
            p, v, a = sim.read_soa()
            assert np.array_equal(p, pos) and np.array_equal(v, vel) and np.all(a == 0), n
            only = np.full((n, 3), np.nan, np.float32)  # one field alone
            st = pu.load_library().nbody_read_soa(sim._h, None, only.ctypes.data_as(fp), None, n)
            assert st == 0 and np.array_equal(only, vel), n


@pytest.mark.parametrize("n", [1, 300, 233017])
def test_records(gpu, n):
    pu = gpu
    pos, vel, mass = _state(n, 2)
    with pu.NBodySim(pu.default_config()) as sim:
        sim.init_soa(pos, vel, mass)
        parts = np.zeros(n, pu.PARTICLE_DTYPE)
        parts["colour"] = 0.25
        sim.read_particles(parts, pu.FIELD_VELOCITY | pu.FIELD_MASS)
        assert np.array_equal(parts["velocity"], vel.astype(np.float64)) and np.array_equal(parts["mass"], mass)
        assert np.all(parts["position"] == 0) and np.all(parts["colour"] == 0.25)
        sim.read_particles(parts, pu.FIELD_POSITION)
        assert np.array_equal(parts["position"], pos)


def test_batch_reads_of_many_sizes(gpu):
    pu = gpu
    sets = [_state(n, 3) for n in (300, 1, 20000, 256, 240000, 257)]
    with pu.Batch(pu.default_config(), 280000) as b:
        ids = [b.add(*s) for s in sets]
        for k in (0, 4, 1, 2, 5, 3, 4):
            p, v, _ = b.read(ids[k])
            assert np.array_equal(p, sets[k][0]) and np.array_equal(v, sets[k][1])
