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
