"""Propagation with and without staged environments: the same bits on both sides of the population
size that the source puts between the two, for every model and precision."""
import pathlib
import re

import numpy as np
import pytest

import ladds_amd as la

pytestmark = pytest.mark.gpu

SOURCE = pathlib.Path(la.__file__).parent / "csrc" / "propagate.hip"
EDGE = int(re.search(r"kStagedObjects = (\d+);", SOURCE.read_text()).group(1))


def _state(pop, precision, mask, n):
    part = la.Population(**{k: x[:n].copy() for k, x in pop.__dict__.items()})
    with la.Engine(la.EngineConfig(precision=precision, components=mask, cutoff_km=10.0)) as eng:
        eng.set_objects(part)
        eng.propagate(3)
        return eng.state()


@pytest.fixture(scope="module")
def population():
    pop = la.generate_population(1, 0x1ADD5 + 91, EDGE + 1)
    # wavefronts with and without an object that feels the Keplerian term only
    pop.activity[100::640] = la.EVASIVE_PRESERVING
    return pop


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT, la.SPLIT_ALL32])
@pytest.mark.parametrize("mask", [la.ALL_COMPONENTS, la.KEP | la.J2, la.KEP, la.KEP | la.DRAG | la.SRP,
                                  la.J2 | la.C22 | la.SOL, la.KEP | la.S22 | la.LUN, 0])
def test_staged_and_unstaged_agree(population, precision, mask):
    wide = _state(population, precision, mask, EDGE + 1)
    staged = _state(population, precision, mask, EDGE)
    for a, b in zip(wide, staged):
        assert np.isfinite(a).all() and np.array_equal(a[:EDGE], b)


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT, la.SPLIT_ALL32])
@pytest.mark.parametrize("n", [EDGE, EDGE + 70])
def test_no_force_without_components(precision, n):
    r = np.zeros((n, 3))
    r[:, 0] = np.arange(n)  # (the first one at the origin)
    r[3] = [np.inf, 0.0, 0.0]
    r[5] = [0.0, 1.0e300, -1.0e-200]
    v = np.zeros_like(r)
    v[:, 2] = np.arange(n) * 1.0e-3
    with la.Engine(la.EngineConfig(precision=precision, components=0, cutoff_km=10.0, dt=1.0)) as eng:
        eng.set_objects(rx=r[:, 0], ry=r[:, 1], rz=r[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2], radius_m=np.ones(n))
        eng.propagate(3)
        r1, v1 = eng.state()
    assert np.array_equal(v1, v)
    assert np.array_equal(r1[:, :2], r[:, :2])
    np.testing.assert_allclose(r1[:, 2], r[:, 2] + 3.0 * v[:, 2], rtol=1e-14, atol=1e-14)
