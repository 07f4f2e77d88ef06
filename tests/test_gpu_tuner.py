"""The autotuner times the shapes that change the kernel that runs."""
import numpy as np
import pytest

import ladds_amd as la

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
@pytest.mark.parametrize("scenarios", [1, 4])
@pytest.mark.parametrize("tune_simulate", [0, 1])
def test_sparse_populations(precision, scenarios, tune_simulate):
    """While the sparse pair kernel runs, its workgroup size, LDS share and buckets are its own: the tuner
    returns their defaults.  Chunks (5 shapes), cell sizes (3), plane widths (3), tiles (3), order,
    persistence (and pair streams, plane sizes) remain; ensembles go over them twice."""
    sizes = [5000] * scenarios
    pop, off = la.generate_ensemble(sizes, 77, workload=0)
    with la.Engine(la.EngineConfig(dt=10.0, components=la.KEP | la.J2, precision=precision, cutoff_km=10.0,
                                   threshold_mode=la.THRESHOLD_ABSOLUTE, threshold_km=1.0,
                                   tune_simulate=tune_simulate)) as eng:
        eng.set_objects(pop)
        if scenarios > 1:
            eng.set_scenarios(off)
        before = eng.conjunction_digest()
        t = eng.autotune(repetitions=2)
        assert eng.conjunction_digest() == before
    if t["chunks"] == 1 and not t["persistent"]:
        assert t["workgroups_per_cu"] == 0 and t["row_cells"] == 1 and t["bucket_cells"] == 1
        assert t["tried"] <= (2 * 21 if scenarios > 1 else 16) + 1 + 2 * tune_simulate


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
def test_clustered_populations(precision):
    """The sorting kernel's dimensions are still searched where it runs."""
    rng = np.random.default_rng(5)
    centres = rng.uniform(-1.0, 1.0, (60, 3)) * [7000.0, 3000.0, 3000.0]
    r = np.repeat(centres, 100, axis=0) + rng.uniform(-4.5, 4.5, (6000, 3))
    v = rng.normal(0.0, 0.2, r.shape)
    with la.Engine(la.EngineConfig(dt=10.0, components=0, precision=precision, cutoff_km=10.0,
                                   threshold_mode=la.THRESHOLD_ABSOLUTE, threshold_km=1.0)) as eng:
        eng.set_objects(rx=r[:, 0], ry=r[:, 1], rz=r[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2], radius_m=np.ones(6000))
        before = eng.conjunction_digest()
        t = eng.autotune(repetitions=1)
        assert eng.conjunction_digest() == before and before[0] > 0
        assert t["tried"] > 30 and t["scan_us"] <= t["default_us"]
