"""The loops of ladds_simulate against each other: kernels of a step on one stream or overlapped,
replayed from graphs of one and of several steps, serial and forked."""
import numpy as np
import pytest

import ladds_amd as la

pytestmark = pytest.mark.gpu


def _run(pop, precision, graph, calls, tpcd=1):
    cfg = la.EngineConfig(dt=10.0, components=3, precision=precision, cutoff_km=10.0, log_capacity=1 << 20,
                          threshold_mode=la.THRESHOLD_ABSOLUTE, threshold_km=2.0, step_graph=graph)
    out, it = [], 0
    with la.Engine(cfg) as eng:
        eng.set_objects(pop)
        for steps in calls:
            s = eng.simulate(steps, first_iteration=it, tpcd=tpcd, min_altitude_km=150.0)
            it += steps
            log = eng.fetch_log()
            eng.clear_log()
            order = np.lexsort((log["pair"]["id_b"], log["pair"]["id_a"], log["iteration"]))
            out.append((s["collisions"], s["remaining"], log[order].tobytes()))
            eng.conjunction_digest()  # eager work between the replays
        r, v = eng.state()
    return out, r, v


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
@pytest.mark.parametrize("n,calls", [
    (20000, [33, 34, 41, 8, 50]),   # serial graphs: at, above and below the several-step graph's least length
    (40001, [40, 35]),              # the eager loop overlaps, the graphs are serial
    (262145, [49, 34]),             # both overlap
])
def test_graphs_match_the_eager_loop(precision, n, calls):
    pop = la.generate_population(1, 11, n)
    got, r0, v0 = _run(pop, precision, 0, calls)
    want, r1, v1 = _run(pop, precision, 1, calls)
    assert sum(g[0] for g in got) > 0
    for a, b in zip(got, want):
        assert a == b
    assert np.array_equal(r0, r1) and np.array_equal(v0, v1)


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT])
@pytest.mark.parametrize("tpcd", [1, 2, 3, 5])
@pytest.mark.parametrize("n", [32769, 262145])
def test_serial_and_overlapped_loops_agree(precision, tpcd, n):
    """32,768 objects run on one stream, 32,769 overlapped (262,144 and 262,145: the partition behind
    the propagation, and beside the next): the last one, far from all others, changes nothing else."""
    pop = la.generate_population(1, 12, n)
    r = pop.r()
    far = 60000.0 / np.linalg.norm(r[-1])
    pop.rx[-1], pop.ry[-1], pop.rz[-1] = r[-1] * far
    full, rf, vf = _run(pop, precision, 0, [13, 6], tpcd)
    for name, arr in list(pop.__dict__.items()):
        if isinstance(arr, np.ndarray) and len(arr) == n:
            setattr(pop, name, arr[:-1].copy())
    less, rl, vl = _run(pop, precision, 0, [13, 6], tpcd)
    for a, b in zip(full, less):
        assert a[0] == b[0] and a[1] == b[1] + 1 and a[2] == b[2]
    assert np.array_equal(rf[:-1], rl) and np.array_equal(vf[:-1], vl)
