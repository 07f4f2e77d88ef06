"""The sparse pair kernel (plane groups with an occupancy map) at the edges of its shapes: pair
sets bit-identical to the oracle's, list and digest output, both forms."""
import numpy as np
import pytest

import ladds_amd as la
import oracle_lib as ol
from test_gpu_parity import _pair_equal

pytestmark = pytest.mark.gpu


def _check(eng, radius, threshold, dt=10.0):
    hits, ev = eng.conjunctions()
    cnt, dig, _, _ = eng.conjunction_digest()
    r, v = eng.state()
    oh, oe = ol.pairs(ol.ObjectSet(r, v, radius), ol.functor_cfg(10.0, dt, threshold_mode=1, threshold_km=threshold))
    _pair_equal(ol.sort_pairs(hits), oh)
    _pair_equal(ol.sort_pairs(ev), oe)
    assert cnt == oh.shape[0] and dig == ol.digest(oh)
    return oh.shape[0]


def _engine(precision, threshold):
    return la.Engine(la.EngineConfig(dt=10.0, components=0, precision=precision, cutoff_km=10.0,
                                     threshold_mode=la.THRESHOLD_ABSOLUTE, threshold_km=threshold))


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
@pytest.mark.parametrize("n,half", [(2, 3.0), (63, 20.0), (65, 20.0), (129, 30.0), (1025, 60.0),
                                    (8003, None), (16384, None), (24001, None)])
def test_group_and_workgroup_sizes(precision, n, half):
    """Clouds in a cube, and slabs 220 km thick in x whose planes are as full as those of the
    largest populations (128 and 256 threads, one and two planes per workgroup)."""
    rng = np.random.default_rng(n)
    box = [half] * 3 if half else [110.0, 2600.0, 2600.0]
    r = rng.uniform(-1.0, 1.0, (n, 3)) * box
    v = rng.normal(0.0, 0.3, (n, 3))
    # the last ones share a cell, or face one across the fold of the map (128 x 256 cells)
    r[-1] = r[0] + [0.1, 0.2, -0.1]
    if n > 1000:
        r[-2] = r[1] + [3.0, 1280.0 - 4.0, 2.0]
        r[-3] = r[2] + [-2.0, 5.0, 2560.0 - 3.0]
    radius = np.full(n, 1.0)
    with _engine(precision, 4.0) as eng:
        eng.set_objects(rx=r[:, 0], ry=r[:, 1], rz=r[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2], radius_m=radius)
        assert _check(eng, radius, 4.0) > 0


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
@pytest.mark.parametrize("n,yz", [(6000, 400.0), (5000, 40.0)])
def test_planes_that_outgrow_their_room(precision, n, yz):
    """Objects spread over every plane when the shape is chosen, and all in one plane when the
    scan runs: records inserted and listed in many turns, the pair list emptied many times."""
    rng = np.random.default_rng(n)
    r = np.stack([np.linspace(-8000.0, 8000.0, n), rng.uniform(-yz, yz, n), rng.uniform(-yz, yz, n)], 1)
    v = np.stack([(5.0 - r[:, 0]) / 10.0, rng.normal(0, 0.1, n), rng.normal(0, 0.1, n)], 1)
    radius = np.full(n, 1.0)
    with _engine(precision, 1.0) as eng:
        eng.set_objects(rx=r[:, 0], ry=r[:, 1], rz=r[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2], radius_m=radius)
        eng.propagate(1)
        assert _check(eng, radius, 1.0) > 0


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
def test_scenarios_without_objects(precision):
    rng = np.random.default_rng(4)
    off = np.array([0, 0, 400, 400, 400, 1100, 1100])
    r, v = rng.uniform(-30.0, 30.0, (1100, 3)), rng.normal(0.0, 0.2, (1100, 3))
    radius = np.full(1100, 1.0)
    with _engine(precision, 3.0) as eng:
        eng.set_objects(rx=r[:, 0], ry=r[:, 1], rz=r[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2], radius_m=radius)
        eng.set_scenarios(off)
        hits, _ = eng.conjunctions()
    want = set()
    for lo, hi in ((0, 400), (400, 1100)):
        oh, _ = ol.pairs(ol.ObjectSet(r[lo:hi], v[lo:hi], radius[lo:hi]),
                         ol.functor_cfg(10.0, 10.0, threshold_mode=1, threshold_km=3.0))
        want |= {(int(a) + lo, int(b) + lo, float(d)) for a, b, d in zip(oh["idx_a"], oh["idx_b"], oh["d2"])}
    got = [(int(a), int(b), float(d)) for a, b, d in zip(hits["idx_a"], hits["idx_b"], hits["d2"])]
    assert len(got) == len(set(got)) and set(got) == want and len(want) > 50


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
@pytest.mark.parametrize("xbox,clusters,size,chunks,rows", [
    (7000.0, 40, 63, 0, 0),   # 256 threads, 2x2-cell buckets
    (7000.0, 40, 65, 0, 1),   # buckets of one cell: three rows, three buckets each
    (7000.0, 900, 6, 0, 0),   # runs shorter than a wavefront: several clusters per 64 records
    (110.0, 60, 130, 0, 0),   # full planes: 512 or 1024 threads, heaviest plane first
    (110.0, 60, 130, 5, 0),   # a plane's buckets shared by five workgroups
    (0.0, 1, 2100, 0, 0),     # one cell: one plane divided over workgroups
])
def test_crowded_cells(precision, xbox, clusters, size, chunks, rows):
    """Clusters within the search radius of themselves, on the borders of cells, buckets and folds, with
    a thin background: the walk by whole wavefronts and the walk lane by lane beside it."""
    rng = np.random.default_rng(clusters * 1000 + size)
    cell = 10.0 if precision == la.FP64 else 10.0 * (1.0 + 1e-5) + 0.1
    centres = rng.uniform(-1.0, 1.0, (clusters, 3)) * [xbox, 3000.0, 3000.0]
    border = 2.0 * cell * 2.0 ** rng.integers(0, 6, (clusters, 2))  # corners of two cells up to a whole fold
    at = rng.random(clusters) < 0.7
    centres[at, 1:] = (np.round(centres[at, 1:] / border[at]) * border[at])
    r = np.repeat(centres, size, axis=0) + rng.uniform(-4.5, 4.5, (clusters * size, 3))
    r = np.concatenate([r, rng.uniform(-1.0, 1.0, (500, 3)) * [max(xbox, 10.0), 3000.0, 3000.0]])
    r = r[rng.permutation(len(r))]
    n = len(r)
    v = rng.normal(0.0, 0.2, (n, 3))
    radius = np.full(n, 1.0)
    cfg = la.EngineConfig(dt=10.0, components=0, precision=precision, cutoff_km=10.0, scan_chunks=chunks,
                          threshold_mode=la.THRESHOLD_ABSOLUTE, threshold_km=1.0)
    with la.Engine(cfg) as eng:
        if rows:
            eng.set_tuning(dict(cell_size_km=cell * 1.0001, plane_width_km=cell * 1.0001, plane_bits=7,
                                pair_threads=256, tile_size=8192, chunks=2, workgroups_per_cu=0,
                                row_cells=1, bucket_cells=1))
        eng.set_objects(rx=r[:, 0], ry=r[:, 1], rz=r[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2], radius_m=radius)
        assert _check(eng, radius, 1.0) > 0


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
@pytest.mark.parametrize("n,half", [(230000, 5000.0), (830000, 10000.0)])
def test_planes_for_every_cu(precision, n, half):
    """More full planes than CUs: 256 threads and one plane, or two, per workgroup."""
    rng = np.random.default_rng(n)
    r = rng.uniform(-1.0, 1.0, (n, 3)) * [half, 700.0, 700.0]
    v = rng.normal(0.0, 0.3, (n, 3))
    radius = np.full(n, 1.0)
    with _engine(precision, 4.0) as eng:
        eng.set_objects(rx=r[:, 0], ry=r[:, 1], rz=r[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2], radius_m=radius)
        assert _check(eng, radius, 4.0) > 0


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
def test_full_planes_of_an_uneven_ensemble(precision):
    """One large scenario among small ones: its planes hold many times the mean and stay whole."""
    rng = np.random.default_rng(5)
    sizes = np.array([30000, 600, 0, 900, 1200, 700])
    n = int(sizes.sum())
    r = rng.uniform(-1.0, 1.0, (n, 3)) * [500.0, 300.0, 300.0]
    v = rng.normal(0.0, 0.3, (n, 3))
    radius = np.full(n, 1.0)
    off = np.concatenate([[0], np.cumsum(sizes)])
    with _engine(precision, 4.0) as eng:
        eng.set_objects(rx=r[:, 0], ry=r[:, 1], rz=r[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2], radius_m=radius)
        eng.set_scenarios(off)
        hits, _ = eng.conjunctions()
    want = []
    for a, b in zip(off[:-1], off[1:]):
        oh, _ = ol.pairs(ol.ObjectSet(r[a:b], v[a:b], radius[a:b]),
                         ol.functor_cfg(10.0, 10.0, threshold_mode=1, threshold_km=4.0))
        want += [(int(p["id_a"]) + a, int(p["id_b"]) + a) for p in oh]
    assert len(want) > 0 and sorted(zip(hits["id_a"].tolist(), hits["id_b"].tolist())) == sorted(want)
