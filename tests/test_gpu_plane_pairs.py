"""The sparse pair kernel with two planes per workgroup under the heaviest-first dispatch order and in
ensembles: pair sets equal to the oracle's."""
import numpy as np
import pytest

import ladds_amd as la
import oracle_lib as ol

pytestmark = pytest.mark.gpu


def _tuning(precision, order, ensemble_plane):
    cell = 10.0001 if precision == la.FP64 else 10.1002
    return dict(cell_size_km=cell, plane_width_km=cell, plane_bits=9, pair_threads=256, tile_size=8192, chunks=1,
                workgroups_per_cu=0, plane_order=order, ensemble_plane_objects=ensemble_plane)


def _scan(r, v, precision, off, order, ensemble_plane):
    with la.Engine(la.EngineConfig(dt=10.0, components=0, precision=precision, cutoff_km=10.0,
                                   threshold_mode=la.THRESHOLD_ABSOLUTE, threshold_km=4.0)) as eng:
        eng.set_tuning(_tuning(precision, order, ensemble_plane))
        eng.set_objects(rx=r[:, 0], ry=r[:, 1], rz=r[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2],
                        radius_m=np.ones(len(r)))
        if len(off) > 2:
            eng.set_scenarios(off)
        hits, _ = eng.conjunctions()
        assert eng.conjunction_digest()[0] == len(hits)
    return sorted(zip(hits["id_a"].tolist(), hits["id_b"].tolist(), hits["d2"].tolist()))


def _want(r, v, off):
    out = []
    for a, b in zip(off[:-1], off[1:]):
        oh, _ = ol.pairs(ol.ObjectSet(r[a:b], v[a:b], np.ones(b - a)),
                         ol.functor_cfg(10.0, 10.0, threshold_mode=1, threshold_km=4.0))
        out += [(int(p["id_a"]) + int(a), int(p["id_b"]) + int(a), float(p["d2"])) for p in oh]
    return sorted(out)


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
def test_heaviest_first(precision):
    """2,048 planes of ~405 objects, unevenly filled: runs of eight planes change their places."""
    rng = np.random.default_rng(31)
    r = rng.uniform(-1.0, 1.0, (830000, 3)) * [10000.0, 700.0, 700.0]
    r[:, 0] = np.where(rng.random(len(r)) < 0.1, 0.5 * r[:, 0], r[:, 0])
    v = rng.normal(0.0, 0.3, r.shape)
    off = np.array([0, len(r)])
    want = _want(r, v, off)
    assert len(want) > 0
    for order in (0, 1):
        assert _scan(r, v, precision, off, order, 0) == want


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
@pytest.mark.parametrize("order", [0, 1])
def test_scenarios(precision, order):
    """Eight scenarios of 128 planes of ~550 objects: a workgroup's planes, and the one after them, are
    one scenario's; the last group's next plane is the scenario's first."""
    rng = np.random.default_rng(32)
    sizes = np.array([70000, 69001, 72003, 70000, 66000, 71111, 70000, 69999])
    r = rng.uniform(-1.0, 1.0, (int(sizes.sum()), 3)) * [900.0, 700.0, 700.0]
    v = rng.normal(0.0, 0.3, r.shape)
    off = np.concatenate([[0], np.cumsum(sizes)])
    want = _want(r, v, off)
    assert len(want) > 100
    assert _scan(r, v, precision, off, order, 1024) == want
