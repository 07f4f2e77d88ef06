"""Ensembles of crowded scenarios that lose some or all of their objects: the shape of the pair scan
follows what is left, and the context serves the next population."""
import numpy as np
import pytest

import ladds_amd as la
import oracle_lib as ol

pytestmark = pytest.mark.gpu

R_EARTH = 6378.1363


def _crowd(seed, sizes, altitude):
    """Scenarios that are one cloud each (all within a cell), on the same place."""
    rng = np.random.default_rng(seed)
    n = int(np.sum(sizes))
    r = rng.uniform(-2.0, 2.0, (n, 3)) + [R_EARTH + altitude + 5.0, 5.0, 5.0]
    v = rng.normal(0.0, 0.1, (n, 3))
    return r, v, np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)


def _fill(eng, r, v, off):
    eng.set_objects(rx=r[:, 0], ry=r[:, 1], rz=r[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2], radius_m=np.ones(len(r)))
    eng.set_scenarios(off)


def _want(r, v, off):
    return sum(ol.pairs(ol.ObjectSet(r[a:b], v[a:b], np.ones(b - a)),
                        ol.functor_cfg(10.0, 10.0, threshold_mode=1, threshold_km=1.0))[0].shape[0]
               for a, b in zip(off[:-1], off[1:]))


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
@pytest.mark.parametrize("how", ["burnups", "objects", "simulate"])
@pytest.mark.parametrize("left", [0, 1, 40])
def test_crowded_ensemble_that_empties(precision, how, left):
    r, v, off = _crowd(1, [300, 500, 80], 100.0)
    if left:  # the last ones stay
        r[-left:, 0] += 900.0
    with la.Engine(la.EngineConfig(dt=10.0, components=0, precision=precision, cutoff_km=10.0,
                                   threshold_mode=la.THRESHOLD_ABSOLUTE, threshold_km=1.0)) as eng:
        for _ in range(2):  # emptied, then another population in the same context
            _fill(eng, r, v, off)
            assert len(eng.conjunctions()[0]) == _want(r, v, off) > 0
            if how == "burnups":
                assert eng.delete_burnups(150.0) == len(r) - left
            elif how == "objects":
                assert eng.delete_objects(np.arange(len(r) - left, dtype=np.uint64)) == len(r) - left
            else:
                assert eng.simulate(2, min_altitude_km=150.0)["remaining"] == left
                eng.clear_log()
            assert eng.n == left
            hits, _ = eng.conjunctions()
            n, _, _, _ = eng.conjunction_digest()
            rl, vl = eng.state()
            oh, _ = ol.pairs(ol.ObjectSet(rl, vl, np.ones(left)),
                             ol.functor_cfg(10.0, 10.0, threshold_mode=1, threshold_km=1.0)) if left > 1 else ([], [])
            assert len(hits) == n == len(oh)
