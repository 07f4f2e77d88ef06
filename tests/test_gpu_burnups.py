"""Removal of burnt-up objects flagged and counted on the device: the same objects as the squared
norm's comparison on the host, also behind a running propagation and before a detection."""
import numpy as np
import pytest

import ladds_amd as la
import oracle_lib as ol
from test_gpu_parity import _pair_equal

pytestmark = pytest.mark.gpu

R_EARTH = 6378.1363


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
@pytest.mark.parametrize("n,low", [(1, 0), (1, 1), (2047, 5), (2048, 2048), (2049, 1), (4099, 0), (70001, 900)])
def test_removal_behind_a_step(precision, n, low):
    pop = la.generate_population(0, n, n)
    r = pop.r()
    rng = np.random.default_rng(n)
    doomed = rng.permutation(n)[:low]
    r[doomed] *= (R_EARTH + rng.uniform(20.0, 120.0, (low, 1))) / np.linalg.norm(r[doomed], axis=1)[:, None]
    pop.rx, pop.ry, pop.rz = (r[:, k].copy() for k in range(3))
    with la.Engine(la.EngineConfig(dt=1.0, components=3, precision=precision, cutoff_km=10.0,
                                   threshold_mode=la.THRESHOLD_ABSOLUTE, threshold_km=5.0)) as eng:
        eng.set_objects(pop)
        eng.propagate(1)
        r1, _ = eng.state()
        limit = (150.0 + R_EARTH) ** 2
        r2 = (r1[:, 0] * r1[:, 0] + r1[:, 1] * r1[:, 1]) + r1[:, 2] * r1[:, 2]
        eng.set_objects(pop)
        eng.propagate(1)  # still running when the removal is called
        removed = eng.delete_burnups(150.0)
        hits, _ = eng.conjunctions()  # follows the compaction on its stream
        rg, vg = eng.state()
        ids = eng.ids()
        keep = np.nonzero(~(r2 < limit))[0]
        assert removed == n - keep.size and eng.n == keep.size
        assert ids.tolist() == keep.tolist()
        assert np.array_equal(rg, r1[keep])
        oh, _ = ol.pairs(ol.ObjectSet(rg, vg, np.asarray(pop.radius_m)[keep], ids=ids),
                         ol.functor_cfg(10.0, 1.0, threshold_mode=1, threshold_km=5.0))
        _pair_equal(ol.sort_pairs(hits), oh)
        assert eng.delete_burnups(150.0) == 0 and eng.n == keep.size
        if keep.size:
            eng.propagate(1)
            assert eng.delete_burnups(1.0e6) == keep.size and eng.n == 0
        assert eng.delete_burnups(150.0) == 0


@pytest.mark.parametrize("pairs", [0, 1, 255, 256, 257, 4097])
def test_pair_lists_around_the_staged_entries(pairs):
    """As many conjunctions as come back with the counters, one fewer and more; a digest between a
    simulation and its fetch leaves the log alone."""
    r = np.zeros((2 * pairs + 4, 3))
    r[:, 0] = np.arange(len(r)) // 2 * 50.0
    r[1::2, 1] = 0.5
    r[2 * pairs:, 1] += 1000.0 * np.arange(4)
    v = np.zeros_like(r)
    v[:, 2] = np.linspace(0.0, 1e-3, len(r))
    with la.Engine(la.EngineConfig(dt=10.0, components=0, cutoff_km=10.0, threshold_mode=la.THRESHOLD_ABSOLUTE,
                                   threshold_km=5.0, log_capacity=8192)) as eng:
        eng.set_objects(rx=r[:, 0], ry=r[:, 1], rz=r[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2],
                        radius_m=np.ones(len(r)))
        for _ in range(2):
            hits, evaded = eng.conjunctions()
            hits = ol.sort_pairs(hits)
            assert len(evaded) == 0
            assert hits["id_a"].tolist() == list(range(0, 2 * pairs, 2))
            assert hits["id_b"].tolist() == list(range(1, 2 * pairs, 2))
        s = eng.simulate(1, first_iteration=0, tpcd=1)
        n, digest, _, _ = eng.conjunction_digest()
        assert n == s["collisions"] == len(eng.fetch_log()) == pairs
        assert digest == ol.digest(hits)
