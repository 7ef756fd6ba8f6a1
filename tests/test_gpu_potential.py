"""The pair potential of the diagnostics: separations from far below to far
above the softening length (the arctangent's argument on both sides of 1),
coincident particles, sizes at the edges of the blocks of 256, and the states
that keep the library's functions (no softening, positions that are not
finite).

Tolerance: each pair's value is within a few units of 2^-53, and a block's 256
pairs and the blocks are added one after another, at most about 600 roundings
for these sizes: 600 x 2^-53 = 7e-14, taken as 1e-13."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def potential(pos, mass, law_r, soft):
    L = np.longdouble
    i, j = np.triu_indices(len(pos), 1)
    p, m = pos.astype(L), mass.astype(L)
    r2 = ((p[i] - p[j]) ** 2).sum(axis=1)
    S = L(soft)
    if not law_r:
        g = 1 / np.sqrt(r2 + S)
    elif soft > 0:
        g = np.arctan2(np.sqrt(S), np.sqrt(r2)) / np.sqrt(S)
    else:
        g = np.where(r2 > 0, 1 / np.sqrt(np.where(r2 > 0, r2, 1)), 0)
    return float(-(m[i] * m[j] * g).sum())


@pytest.mark.parametrize("law", ["R", "P"])
@pytest.mark.parametrize("n,soft", [(2, 1e-12), (2, 1e-2), (2, 1e6), (3, 1.0), (255, 1e-4), (256, 1.0), (257, 1e4),
                                    (511, 1e-2), (513, 1e-8)])
def test_potential_matches_extended_precision(gpu, law, n, soft):
    pu = gpu
    rng = np.random.default_rng(0xD1A6 + n)
    pos = (rng.normal(size=(n, 3)) * 10.0 ** rng.uniform(-3, 3, size=(n, 1))).astype(np.float32)
    if n > 2:
        pos[n // 2] = pos[0]  # coincident, not the same particle
    mass = rng.uniform(0.5, 1.5, n)
    cfg = pu.default_config(method=pu.METHOD_DIRECT, law=pu.LAW_R if law == "R" else pu.LAW_P, softening=soft)
    with pu.NBodySim(cfg) as sim:
        sim.init_soa(pos, np.zeros_like(pos), mass)
        got = sim.diagnostics()["potential"]
    ref = potential(pos, mass, law == "R", soft)
    assert abs(got - ref) <= 1e-13 * abs(ref), (got, ref)


def test_potential_without_softening_and_with_an_infinite_position(gpu):
    pu = gpu
    rng = np.random.default_rng(5)
    pos = rng.normal(size=(300, 3)).astype(np.float32)
    mass = rng.uniform(0.5, 1.5, 300)
    cfg = pu.default_config(method=pu.METHOD_DIRECT, law=pu.LAW_R, softening=0.0)
    with pu.NBodySim(cfg) as sim:
        sim.init_soa(pos, np.zeros_like(pos), mass)
        got = sim.diagnostics()["potential"]
        ref = potential(pos, mass, True, 0.0)
        assert abs(got - ref) <= 1e-13 * abs(ref), (got, ref)
    # a particle at infinity adds nothing to the others' potential, a NaN makes it NaN
    for law in (pu.LAW_R, pu.LAW_P):
        cfg = pu.default_config(method=pu.METHOD_DIRECT, law=law, softening=0.25)
        for bad, expect in ((np.inf, potential(np.delete(pos, 270, 0), np.delete(mass, 270), law == pu.LAW_R, 0.25)),
                            (np.nan, np.nan)):
            odd = pos.copy()
            odd[270, 1] = bad
            with pu.NBodySim(cfg) as sim:
                sim.init_soa(odd, np.zeros_like(odd), mass)
                got = sim.diagnostics()["potential"]
            assert np.isnan(got) if np.isnan(expect) else abs(got - expect) <= 1e-13 * abs(expect)
