"""What is timed: the work that programs have this engine do, through its public entry points.

Five kinds of pass:

step       one iteration of a hand-driven loop (integrate, remove burn-ups, detect, refresh the
           objects of the pairs found), as a host program that keeps its own loop calls it
simulate   a stretch of the simulation loop up to the next output, then the pair log and the
           particle records that are written there
screen     one conjunction screening of a snapshot, counts and digest only
propagate  propagation alone over many steps, then the state
gradient   propagation with its gradient (orbit fitting): final state, and the gradients of a
           squared-distance loss with respect to the initial state and the drag coefficient

Sizes are those of the repository's workloads (16,384 objects; 1,048,576 objects with a
debris tail; clustered constellations; an ensemble of 1,024-65,536 objects per scenario; 4,096
objects differentiated over a day of 60 s steps) and odd ones between them.
"""
import math

import numpy as np
import torch

import ladds_amd as la
from ladds_amd import adjoint

MIN_ALTITUDE = 150.0  # km, below which the simulation loop removes objects
KEPLER_J2 = la.KEP | la.J2
R_EARTH = 6378.1363

# A shape that autotuning picked for the 1,048,576-object split workload and that a program
# keeps from then on (set_tuning), as a calibrated configuration is kept.
CALIBRATED = {"cell_size_km": 10.1002, "plane_width_km": 10.1002, "plane_bits": 10, "pair_threads": 256,
              "tile_size": 8192, "chunks": 1, "workgroups_per_cu": 0, "plane_order": 0, "row_cells": 2,
              "bucket_cells": 1, "pair_streams": 2}


def listed():
    return [
        # The smallest call: one iteration of a hand-driven loop on the 16,384-object workload
        # (Kepler + J2), where launches and latency count.
        {"name": "step 16384 fp64", "kind": "step", "n": 16384, "model": "j2", "precision": "fp64", "burnups": False},
        # The same loop on a catalogue-sized population with the full force model, burn-ups removed
        # in every iteration as the simulation loop does.
        {"name": "step 100003 split", "kind": "step", "n": 100003, "model": "full", "precision": "split",
         "burnups": True},
        # The 16,384-object workload as one call: 100 iterations with a detection in each.
        {"name": "simulate 16384 fp64", "kind": "simulate", "n": 16384, "model": "j2", "precision": "fp64",
         "steps": 100, "tpcd": 1, "cutoff": 10.0, "scenarios": 0, "sizes": 0, "graph": 0, "tuned": False},
        # Default cutoff (80 km), a detection every 10 iterations, radius-scaled threshold and
        # evasive objects: an ordinary long-term run with defaults.
        {"name": "simulate 65521 wide", "kind": "simulate", "n": 65521, "model": "full", "precision": "fp64",
         "steps": 400, "tpcd": 10, "cutoff": 80.0, "scenarios": 0, "sizes": 0, "graph": 0, "tuned": False},
        # The headline workload, both forms, over four hours (three quarters of an hour for
        # FP64): 1,048,576 objects, full force model, detection in every iteration.
        {"name": "simulate 1M split", "kind": "simulate", "n": 1048576, "model": "full", "precision": "split",
         "steps": 1440, "tpcd": 1, "cutoff": 10.0, "scenarios": 0, "sizes": 0, "graph": 0, "tuned": True},
        {"name": "simulate 1M fp64", "kind": "simulate", "n": 1048576, "model": "full", "precision": "fp64",
         "steps": 270, "tpcd": 1, "cutoff": 10.0, "scenarios": 0, "sizes": 0, "graph": 0, "tuned": False},
        # Monte Carlo: 64 scenarios of 1,024-65,536 objects, steps replayed from a HIP graph.
        {"name": "ensemble 64", "kind": "simulate", "n": 0, "model": "full", "precision": "split", "steps": 300,
         "tpcd": 1, "cutoff": 10.0, "scenarios": 64, "sizes": 3, "graph": 1, "tuned": False},
        # Screening of clustered constellations (60% of the objects sit in 4,668 slots).
        {"name": "screen 1M clustered", "kind": "screen", "n": 1048576, "population": 2, "precision": "split",
         "cutoff": 5.0, "threshold": 0.5},
        # Propagation between outputs without detections, and a small group over a long span
        # (one wavefront per compute unit or less: a chain of dependent steps).
        {"name": "propagate 250007 fp64", "kind": "propagate", "n": 250007, "model": "full", "precision": "fp64",
         "steps": 1000},
        {"name": "propagate 4099 split", "kind": "propagate", "n": 4099, "model": "full", "precision": "split",
         "steps": 1500},
        # Orbit fitting: the 4,096-object workload over a day, and many objects over an hour.
        {"name": "gradient 4096 day", "kind": "gradient", "n": 4096, "steps": 1440, "dt": 60.0, "every": 64},
        {"name": "gradient 50021 hour", "kind": "gradient", "n": 50021, "steps": 60, "dt": 60.0, "every": 16},
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "simulate", "simulate", "ensemble", "screen", "propagate", "gradient"])
    precision = rng.choice(["fp64", "split"])
    model = rng.choice(["full", "full", "j2"])
    if kind == "step":
        return {"kind": "step", "n": _spread(rng, 4096, 262144), "model": model, "precision": precision,
                "burnups": rng.random() < 0.5}
    if kind == "simulate":
        n = _spread(rng, 16384, 1048576)
        steps = min(_spread(rng, 20, 1440), max(20, int(3e8 / n)))
        wide = n <= 200000 and rng.random() < 0.4
        return {"kind": "simulate", "n": n, "model": model, "precision": precision, "steps": steps,
                "tpcd": rng.choice([3, 10]) if wide else rng.choice([1, 1, 2]), "cutoff": 80.0 if wide else 10.0,
                "scenarios": 0, "sizes": 0, "graph": int(rng.random() < 0.2),
                "tuned": precision == "split" and n > 700000}
    if kind == "ensemble":
        return {"kind": "simulate", "n": 0, "model": model, "precision": precision, "steps": _spread(rng, 50, 300),
                "tpcd": 1, "cutoff": 10.0, "scenarios": rng.randint(12, 64), "sizes": rng.randint(0, 999),
                "graph": int(rng.random() < 0.7), "tuned": False}
    if kind == "screen":
        population = rng.choice([1, 2])
        cutoff = rng.choice([5.0, 10.0]) if population == 1 else 5.0
        return {"kind": "screen", "n": _spread(rng, 131072, 1048576), "population": population,
                "precision": precision, "cutoff": cutoff, "threshold": rng.choice([0.5, 1.0]) if cutoff > 5.0 else 0.5}
    if kind == "propagate":
        n = _spread(rng, 1024, 1048576)
        return {"kind": "propagate", "n": n, "model": model, "precision": precision,
                "steps": min(_spread(rng, 100, 1500), max(50, int(2.5e8 / n)))}
    n = _spread(rng, 256, 65536)
    return {"kind": "gradient", "n": n, "steps": min(_spread(rng, 16, 1440), max(16, int(5e6 / n))),
            "dt": rng.choice([10.0, 60.0]), "every": rng.choice([16, 64, 100])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _sizes(case):
    """Scenario sizes of an ensemble: log-uniform 1,024-65,536 objects."""
    rng = np.random.default_rng(case["sizes"])
    return np.exp(rng.uniform(math.log(1024), math.log(65536), case["scenarios"])).astype(np.int64)


def _in_orbit(workload, seed, n, perigee_km):
    """n objects of a seeded population whose perigee is above `perigee_km`: the ones that stay in
    orbit over the span, where no burn-up removal runs beside the propagation."""
    pop = la.generate_population(workload, seed, n + n // 4 + 64)
    r, v = pop.r(), pop.v()
    rn = np.linalg.norm(r, axis=1)
    mu = 398600.4418
    a = 1.0 / (2.0 / rn - np.einsum("ij,ij->i", v, v) / mu)
    h = np.cross(r, v)
    e = np.sqrt(np.maximum(0.0, 1.0 - np.einsum("ij,ij->i", h, h) / (mu * a)))
    keep = np.nonzero(a * (1.0 - e) > R_EARTH + perigee_km)[0][:n]
    for name, arr in list(pop.__dict__.items()):
        setattr(pop, name, arr[keep].copy())
    pop.id = np.arange(n, dtype=np.uint64)
    return pop


def _crossing_pairs(pop, seed, count):
    """The last `count` objects moved 0.3-0.9 km above `count` others, their velocities turned
    by 1-5 degrees: encounters in the first iteration."""
    rng = np.random.default_rng(seed)
    n = pop.n
    base = rng.permutation(n - count)[:count]
    r, v = pop.r()[base], pop.v()[base]
    u = r / np.linalg.norm(r, axis=1)[:, None]
    ang = np.deg2rad(rng.uniform(1.0, 5.0, count))[:, None]
    turned = (v * np.cos(ang) + np.cross(u, v) * np.sin(ang)
              + u * np.sum(u * v, axis=1)[:, None] * (1.0 - np.cos(ang)))
    moved = r + u * rng.uniform(0.3, 0.9, count)[:, None]
    for k, name in enumerate(("rx", "ry", "rz")):
        getattr(pop, name)[n - count:] = moved[:, k]
    for k, name in enumerate(("vx", "vy", "vz")):
        getattr(pop, name)[n - count:] = turned[:, k]


def _population(case, seed):
    kind = case["kind"]
    if kind == "gradient":
        return _in_orbit(0, seed, case["n"], 300.0)
    if kind == "propagate":
        return _in_orbit(1, seed, case["n"], 350.0)
    if kind == "screen":
        pop = la.generate_population(case["population"], seed, case["n"])
        if case["population"] != 2:
            _crossing_pairs(pop, seed, 64)
        pop.id = np.random.default_rng(seed).permutation(pop.n).astype(np.uint64)  # catalogue numbers
        return pop
    if case.get("scenarios"):
        return la.generate_ensemble(_sizes(case), seed << 8, workload=0)[0]
    pop = la.generate_population(1 if case["model"] == "full" else 0, seed, case["n"])
    _crossing_pairs(pop, seed, 64)
    if case.get("cutoff") == 80.0:  # a third of the objects can evade
        pop.activity = (np.random.default_rng(seed + 1).random(pop.n) < 0.33).astype(np.int32)
    return pop


def _config(case):
    kw = {"dt": 10.0, "precision": la.SPLIT if case["precision"] == "split" else la.FP64,
          "components": KEPLER_J2 if case.get("model") == "j2" else la.ALL_COMPONENTS,
          "cutoff_km": case.get("cutoff", 10.0)}
    if case.get("cutoff") == 80.0:
        kw.update(collision_distance_factor=500.0, evasion_cutoff_km=1.0)
    else:
        kw.update(threshold_mode=la.THRESHOLD_ABSOLUTE, threshold_km=case.get("threshold", 1.0))
    if case["kind"] == "simulate":
        kw.update(step_graph=case["graph"], log_capacity=1 << 22)
    return la.EngineConfig(**kw)


def prepare(case, seed):
    pop = _population(case, seed)
    if case["kind"] == "gradient":
        dev = torch.device("cuda:0")
        to = lambda x: torch.tensor(np.ascontiguousarray(x), dtype=torch.float64, device=dev)  # noqa: E731
        plan = adjoint.AdjointPlan(pop.n, case["steps"], case["dt"], components=la.ALL_COMPONENTS,
                                   checkpoint_every=case["every"])
        r0, v0, bc = (to(x).requires_grad_() for x in (pop.r(), pop.v(), pop.bc_inv))
        aom, cr = to(pop.aom), to(pop.cr)
        with torch.no_grad():
            nominal, _ = adjoint.propagate(r0, v0, bc, plan, aom=aom, cr=cr)
        noise = to(np.random.default_rng(seed).normal(0.0, 0.1, (pop.n, 3)))  # observations: 100 m
        return {"kind": "gradient", "plan": plan, "r0": r0, "v0": v0, "bc": bc, "aom": aom, "cr": cr,
                "target": nominal + noise}
    eng = la.Engine(_config(case))
    if case.get("tuned"):
        eng.set_tuning(CALIBRATED)
    eng.set_objects(pop)
    if case.get("scenarios"):
        eng.set_scenarios(np.concatenate([[0], np.cumsum(_sizes(case))]))
    tables = ()
    if case["kind"] == "simulate":
        tables = np.zeros((pop.n, 3), np.float32), np.zeros((pop.n, 3), np.float32), np.zeros(pop.n, np.int64)
    return {"kind": case["kind"], "eng": eng, "case": case, "iteration": 0, "tables": tables}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _by_ids(pairs):
    return pairs[np.argsort((pairs["id_a"] << np.uint64(32)) | pairs["id_b"])]


def _rows(count, unit):
    """Rows of the table that `count` entries are kept in: whole blocks of `unit`."""
    return max(1, -(-count // unit)) * unit


def _table(pairs, rows):
    """The pairs at the start of a table of `rows` entries, column by column."""
    out = np.zeros(rows, pairs.dtype)
    out[:len(pairs)] = pairs
    return out


def _columns(pairs):
    return {"id_a": pairs["id_a"].astype(np.int64), "id_b": pairs["id_b"].astype(np.int64), "d2": pairs["d2"],
            "mid": pairs["mid"]}


def _digest(d):
    return np.array(d, np.uint64).view(np.int64)


def run(state):
    if state["kind"] == "gradient":
        s = state
        rT, vT = adjoint.propagate(s["r0"], s["v0"], s["bc"], s["plan"], aom=s["aom"], cr=s["cr"])
        loss = ((rT - s["target"]) ** 2).sum()
        g_r, g_v, g_bc = torch.autograd.grad(loss, (s["r0"], s["v0"], s["bc"]))
        return {"r": rT.detach(), "v": vT.detach(), "g_r": g_r, "g_v": g_v, "g_bc": g_bc}
    eng, case = state["eng"], state["case"]
    if state["kind"] == "step":
        eng.propagate(1)
        removed = eng.delete_burnups(MIN_ALTITUDE) if case["burnups"] else 0
        hits, evaded = eng.conjunctions()
        hits = _by_ids(hits)
        r, v = eng.gather_state(np.concatenate([hits["idx_a"], hits["idx_b"]]))
        rows = _rows(len(hits), 256)
        rv = np.zeros((2, 2, rows, 3))
        rv[:, 0, :len(hits)] = r[:len(hits)], v[:len(hits)]
        rv[:, 1, :len(hits)] = r[len(hits):], v[len(hits):]
        return {"removed": removed, "hits": _columns(_table(hits, rows)), "evasions": len(evaded), "r": rv[0],
                "v": rv[1]}
    if state["kind"] == "screen":
        n, digest, ne, edigest = eng.conjunction_digest()
        return {"collisions": n, "digest": _digest(digest), "evasions": ne, "edigest": _digest(edigest)}
    if state["kind"] == "propagate":
        eng.propagate(case["steps"])
        r, v = eng.state()
        return {"r": r, "v": v}
    stats = eng.simulate(case["steps"], first_iteration=state["iteration"], tpcd=case["tpcd"],
                         min_altitude_km=MIN_ALTITUDE)
    state["iteration"] += case["steps"]
    log = eng.fetch_log()
    eng.clear_log()
    log = log[np.lexsort((log["pair"]["id_b"], log["pair"]["id_a"], log["iteration"]))]
    log = _table(log, _rows(len(log), 65536))
    # the program's own tables of the initial objects: the remaining ones first
    for table, record in zip(state["tables"], eng.particle_records()):
        table[:len(record)] = record
        table[len(record):] = 0
    return {"collisions": stats["collisions"], "evasions": stats["evasions"], "candidates": stats["candidates"],
            "remaining": stats["remaining"], "iteration": log["iteration"].astype(np.int64),
            "evaded": log["evaded"].astype(np.int64), "scenario": log["scenario"].astype(np.int64),
            "pairs": _columns(log["pair"]), "pos": state["tables"][0], "vel": state["tables"][1],
            "ids": state["tables"][2]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    full = case.get("model", "full") == "full"
    flops_step = 809.0 if full else 120.0  # Yoshida step (three force evaluations) of one object
    params = (16 if case.get("precision") == "fp64" else 12) if full else 0
    # detection: the objects' positions written in cell order and read back
    detect = 2 * (32 if case.get("precision") == "fp64" else 16)
    kind, n = case["kind"], case["n"]
    if kind == "gradient":
        s = case["steps"]
        # state, parameters and targets in, final state and gradients out; the reverse sweep
        # recomputes the trajectory and costs about two evaluations per kick
        return {"bytes": n * (48 + 24 + 24 + 48 + 56), "flops": 4.0 * 809.0 * n * s}
    if kind == "propagate":
        return {"bytes": n * (96 + params), "flops": flops_step * n * case["steps"]}
    if kind == "screen":
        return {"bytes": n * (24 + detect), "flops": 100.0 * n}
    if kind == "step":
        return {"bytes": n * (96 + params + detect), "flops": flops_step * n}
    if case["scenarios"]:
        n = int(_sizes(case).sum())
    s = case["steps"]
    return {"bytes": n * ((96 + params) * s + detect * (s // case["tpcd"]) + 28), "flops": flops_step * n * s}


# ---------------------------------------------------------------------------
# the same results in 64 bits by plain torch
# ---------------------------------------------------------------------------
_MU, _J2 = 398600.4418, 1.0826266835531513e-3
_C22, _S22 = 1.574460374564035e-6, -9.03803806638557e-7
_GM_SUN, _GM_MOON, _AU, _P_SUN, _OMEGA = 1.32712440018e11, 4902.800066, 149597870.7, 4.56e-6, 7.2921158553e-5
_H0 = [0, 25, 30, 40, 50, 60, 70, 80, 90, 100, 110, 120, 130, 140, 150, 180, 200, 250, 300, 350, 400, 450, 500, 600,
       700, 800, 900, 1000]
_RHO = [1.225, 3.899e-2, 1.774e-2, 3.972e-3, 1.057e-3, 3.206e-4, 8.770e-5, 1.905e-5, 3.396e-6, 5.297e-7, 9.661e-8,
        2.438e-8, 8.484e-9, 3.845e-9, 2.070e-9, 5.464e-10, 2.789e-10, 7.248e-11, 2.418e-11, 9.518e-12, 3.725e-12,
        1.585e-12, 6.967e-13, 1.454e-13, 3.614e-14, 1.170e-14, 5.245e-15, 3.019e-15]
_SCALE = [7.249, 6.349, 6.682, 7.554, 8.382, 7.714, 6.549, 5.799, 5.382, 5.877, 7.263, 9.473, 12.636, 16.149, 22.523,
          29.740, 37.105, 45.546, 53.628, 53.298, 58.515, 60.828, 63.822, 71.835, 88.667, 124.64, 181.05, 268.00]


def _sun_moon(t):
    """Low-precision solar and lunar positions [km] (Montenbruck & Gill, eq. 3.46-3.50)."""
    deg = math.pi / 180.0
    sec, sin, cos = deg / 3600.0, math.sin, math.cos
    eps = 0.40909280422232897
    T = t / 3155760000.0
    M = (357.5256 + 35999.049 * T) * deg
    L = 282.9400 * deg + M + (6892.0 * sin(M) + 72.0 * sin(2 * M)) * sec
    r = (149.619 - 2.499 * cos(M) - 0.021 * cos(2 * M)) * 1e6
    sun = (r * cos(L), r * sin(L) * cos(eps), r * sin(L) * sin(eps))
    L0 = (218.31617 + 481267.88088 * T - 1.3972 * T) * deg
    l, lp = (134.96292 + 477198.86753 * T) * deg, (357.52543 + 35999.04944 * T) * deg  # noqa: E741
    F, D = (93.27283 + 483202.01873 * T) * deg, (297.85027 + 445267.11135 * T) * deg
    dlam = (22640 * sin(l) + 769 * sin(2 * l) - 4586 * sin(l - 2 * D) + 2370 * sin(2 * D) - 668 * sin(lp)
            - 412 * sin(2 * F) - 212 * sin(2 * l - 2 * D) - 206 * sin(l + lp - 2 * D) + 192 * sin(l + 2 * D)
            - 165 * sin(lp - 2 * D) + 148 * sin(l - lp) - 125 * sin(D) - 110 * sin(l + lp) - 55 * sin(2 * F - 2 * D))
    lam = L0 + dlam * sec
    beta = (18520 * sin(F + lam - L0 + (412 * sin(2 * F) + 541 * sin(lp)) * sec) - 526 * sin(F - 2 * D)
            + 44 * sin(l + F - 2 * D) - 31 * sin(-l + F - 2 * D) - 25 * sin(-2 * l + F) - 23 * sin(lp + F - 2 * D)
            + 21 * sin(-l + F) + 11 * sin(-lp + F - 2 * D)) * sec
    r = (385000 - 20905 * cos(l) - 3699 * cos(2 * D - l) - 2956 * cos(2 * D) - 570 * cos(2 * l)
         + 246 * cos(2 * l - 2 * D) - 205 * cos(lp - 2 * D) - 171 * cos(l + 2 * D) - 152 * cos(l + lp - 2 * D))
    x, y, z = r * cos(lam) * cos(beta), r * sin(lam) * cos(beta), r * sin(beta)
    moon = (x, y * cos(eps) - z * sin(eps), y * sin(eps) + z * cos(eps))
    return sun, moon


class _Model:
    """Acceleration of all objects (rows of (n, 3) tensors) at time t."""

    def __init__(self, full, drag, srp, dev):
        self.full, self.drag, self.srp, self.dev = full, drag, srp, dev
        t = lambda x: torch.tensor(x, dtype=torch.float64, device=dev)  # noqa: E731
        self.h0, self.rho, self.scale = t([float(h) for h in _H0]), t(_RHO), t(_SCALE)
        self.j2 = t([1.0, 1.0, 3.0])

    def __call__(self, r, v, t):
        r2 = (r * r).sum(1, keepdim=True)
        rn = r2.sqrt()
        z2 = 5.0 * r[:, 2:] ** 2 / r2
        acc = -_MU * r / (r2 * rn) - 1.5 * _J2 * _MU * R_EARTH**2 / (r2 * r2 * rn) * r * (self.j2 - z2)
        if not self.full:
            return acc
        vec = lambda x: torch.tensor(x, dtype=torch.float64).to(self.dev)  # noqa: E731
        # C22, S22: U = (kc (x^2 - y^2) + ks x y) / r^5 in the Earth-fixed frame
        th = math.fmod(4.894961212823756 + _OMEGA * t, 2.0 * math.pi)
        c, s = math.cos(th), math.sin(th)
        kc, ks = 3.0 * _MU * R_EARTH**2 * _C22, 6.0 * _MU * R_EARTH**2 * _S22
        x, y = c * r[:, 0] + s * r[:, 1], c * r[:, 1] - s * r[:, 0]
        i5 = (1.0 / (r2 * r2 * rn))[:, 0]
        gx, gy = (2 * kc * x + ks * y) * i5, (ks * x - 2 * kc * y) * i5
        q = 5.0 * (kc * (x * x - y * y) + ks * x * y) * i5 / r2[:, 0]
        acc = acc + torch.stack([c * gx - s * gy, s * gx + c * gy, torch.zeros_like(gx)], 1) - q[:, None] * r
        # third bodies
        sun, moon = _sun_moon(t)
        S, Mo = vec(sun), vec(moon)
        ds, dm = S - r, Mo - r
        is3, im3 = (ds * ds).sum(1, keepdim=True) ** -1.5, (dm * dm).sum(1, keepdim=True) ** -1.5
        s2, m2 = sum(a * a for a in sun), sum(a * a for a in moon)
        indirect = [_GM_SUN * a / (s2 * math.sqrt(s2)) + _GM_MOON * b / (m2 * math.sqrt(m2))
                    for a, b in zip(sun, moon)]
        acc = acc + _GM_SUN * is3 * ds + _GM_MOON * im3 * dm - vec(indirect)
        # solar radiation pressure outside the Earth's cylindrical shadow
        rs = r @ S
        dark = (rs < 0.0) & (r2[:, 0] - rs * rs / s2 < R_EARTH**2)
        acc = acc - torch.where(dark, 0.0, self.srp)[:, None] * is3 * ds
        # drag: exponential atmosphere that turns with the Earth
        h = rn[:, 0] - R_EARTH
        row = (torch.searchsorted(self.h0, h.detach().contiguous(), right=True) - 1).clamp(min=0)
        rho = self.rho[row] * torch.exp(-(h - self.h0[row]) / self.scale[row])
        w = torch.stack([v[:, 0] + _OMEGA * r[:, 1], v[:, 1] - _OMEGA * r[:, 0], v[:, 2]], 1)
        return acc + (self.drag * rho * w.norm(dim=1))[:, None] * w


def _yoshida(model, r, v, steps, dt, burn_r2=0.0):
    """`steps` fourth-order steps (Yoshida 1990); with burn_r2, objects below it stop for good."""
    cb = 2.0 ** (1.0 / 3.0)
    w1, w0 = 1.0 / (2.0 - cb), -cb / (2.0 - cb)
    c, d = (w1 / 2, (w0 + w1) / 2, (w0 + w1) / 2, w1 / 2), (w1, w0, w1)
    alive = torch.ones(r.shape[0], dtype=torch.bool, device=r.device)
    for s in range(steps):
        r0, v0, tau = r, v, 0.0
        for k in range(3):
            r = r + (c[k] * dt) * v
            tau += c[k]
            v = v + (d[k] * dt) * model(r, v, s * dt + tau * dt)
        r = r + (c[3] * dt) * v
        if burn_r2:
            r, v = torch.where(alive[:, None], r, r0), torch.where(alive[:, None], v, v0)
            alive = alive & ~((r * r).sum(1) < burn_r2)
    return r, v, alive


def _close_pairs(r, v, cutoff, dt, threshold):
    """Index pairs within `cutoff` whose closest approach in the last dt seconds is below
    `threshold`, with the squared distance and the midpoint there."""
    found, n = [], r.shape[0]
    for lo in range(0, n, 1024):
        d2 = sum((r[lo:lo + 1024, k, None] - r[None, :, k]) ** 2 for k in range(3))
        i, j = torch.nonzero(d2 <= cutoff * cutoff, as_tuple=True)
        found.append(torch.stack([i + lo, j])[:, i + lo < j])
    i, j = torch.cat(found, 1)
    dr, dv = (r[i] - v[i] * dt) - (r[j] - v[j] * dt), v[i] - v[j]
    t = (-(dr * dv).sum(1) / (dv * dv).sum(1)).clamp(0.0, dt)[:, None]
    gap = dr + dv * t
    d2 = (gap * gap).sum(1)
    keep = d2 <= threshold * threshold
    mid = (r[j] - v[j] * dt) + v[j] * t + 0.5 * gap
    return i[keep], j[keep], d2[keep], mid[keep]


def exact(case, seed):
    kind = case["kind"]
    if kind == "screen" or case["n"] * case.get("steps", 1) > 2e9:
        return None
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    pop = _population_for_exact(case, seed)
    to = lambda x: torch.tensor(np.ascontiguousarray(x), dtype=torch.float64, device=dev)  # noqa: E731
    r, v = to(pop["r"]), to(pop["v"])
    drag, srp = -0.5e3 * to(pop["bc_inv"]), _P_SUN * 1e3 * _AU**2 * to(pop["cr"]) * to(pop["aom"])
    full = case.get("model", "full") == "full"
    if kind == "gradient":
        bc = to(pop["bc_inv"])
        for x in (r, v, bc):
            x.requires_grad_()
        rT, vT, _ = _yoshida(_Model(True, -0.5e3 * bc, srp, dev), r, v, case["steps"], case["dt"])
        noise = to(np.random.default_rng(seed).normal(0.0, 0.1, tuple(r.shape)))
        loss = ((rT - (rT.detach() + noise)) ** 2).sum()
        g_r, g_v, g_bc = torch.autograd.grad(loss, (r, v, bc))
        return {"r": rT.detach(), "v": vT.detach(), "g_r": g_r, "g_v": g_v, "g_bc": g_bc}
    model = _Model(full, drag, srp, dev)
    burn = (R_EARTH + MIN_ALTITUDE) ** 2
    if kind == "propagate":
        r, v, _ = _yoshida(model, r, v, case["steps"], 10.0)
        return {"r": r, "v": v}
    if kind == "step":
        r, v, alive = _yoshida(model, r, v, 1, 10.0, burn if case["burnups"] else 0.0)
        i, j, d2, mid = _close_pairs(r[alive], v[alive], 10.0, 10.0, 1.0)
        ids = torch.arange(len(alive), device=dev)[alive]
        order = torch.argsort(ids[i] * (1 << 32) + ids[j])
        rows = _rows(len(order), 256)
        fill = lambda x: torch.cat([x, x.new_zeros((rows - len(x), *x.shape[1:]))])  # noqa: E731
        ra, va = r[alive], v[alive]
        return {"removed": None, "evasions": None,
                "hits": {"id_a": None, "id_b": None, "d2": fill(d2[order]), "mid": fill(mid[order])},
                "r": torch.stack([fill(ra[i[order]]), fill(ra[j[order]])]),
                "v": torch.stack([fill(va[i[order]]), fill(va[j[order]])])}
    r, v, alive = _yoshida(model, r, v, case["steps"], 10.0, burn)
    r, v = (torch.cat([x[alive], x.new_zeros((int((~alive).sum()), 3))]) for x in (r, v))
    return {"collisions": None, "evasions": None, "candidates": None, "remaining": None, "iteration": None,
            "evaded": None, "scenario": None, "pairs": {"id_a": None, "id_b": None, "d2": None, "mid": None},
            "pos": r, "vel": v, "ids": None}


def _population_for_exact(case, seed):
    """The inputs of prepare() (seeded data, no results of the engine)."""
    pop = _population(case, seed)
    return {"r": pop.r(), "v": pop.v(), "bc_inv": pop.bc_inv, "aom": pop.aom, "cr": pop.cr}
