"""Kernel variants chosen by population size and model give the same bits: propagation with and
without staged environments and with constant or per-lane component masks, and the two forward
passes of the adjoint."""
import numpy as np
import pytest
import torch

import ladds_amd as la

pytestmark = pytest.mark.gpu

EDGE = 32768  # staged environments and the grouped adjoint forward up to here


def _take(pop, n):
    out = pop.copy()
    for k, v in out.__dict__.items():
        setattr(out, k, v[:n].copy())
    return out


def _state(pop, precision, mask, steps=3):
    with la.Engine(la.EngineConfig(precision=precision, components=mask, cutoff_km=10.0)) as eng:
        eng.set_objects(pop)
        eng.propagate(steps)
        return eng.state()


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT, la.SPLIT_ALL32])
@pytest.mark.parametrize("mask", [la.ALL_COMPONENTS, la.KEP | la.J2, la.KEP | la.DRAG | la.SRP])
def test_propagation_variants_agree(precision, mask):
    pop = la.generate_population(1, 0x1ADD5 + 71, EDGE + 1)
    wide = _state(pop, precision, mask)
    staged = _state(_take(pop, EDGE), precision, mask)
    for a, b in zip(wide, staged):
        assert np.array_equal(a[:EDGE], b)
    # an evasivePreserving object takes its wavefront off the constant-mask path: its
    # neighbours keep their bits and it moves under the Keplerian term alone
    pop.activity[100::640] = la.EVASIVE_PRESERVING
    mixed = _state(pop, precision, mask)
    kepler = _state(pop, precision, mask & la.KEP)
    special = pop.activity == la.EVASIVE_PRESERVING
    for a, b, c in zip(mixed, wide, kepler):
        assert np.array_equal(a[~special], b[~special])
        assert np.array_equal(a[special], c[special])


@pytest.mark.parametrize("every", [20, 64])
def test_adjoint_forward_variants_agree(every):
    from ladds_amd import adjoint

    pop = la.generate_population(1, 0x1ADD5 + 72, EDGE + 1)
    t = lambda x: torch.tensor(np.ascontiguousarray(x), dtype=torch.float64, device="cuda:0")

    def run(p):
        plan = adjoint.AdjointPlan(p.n, 70, 30.0, checkpoint_every=every)
        r0, v0, bc = (t(x).requires_grad_() for x in (p.r(), p.v(), p.bc_inv))
        rT, vT = adjoint.propagate(r0, v0, bc, plan, aom=t(p.aom), cr=t(p.cr))
        g = torch.autograd.grad((rT.sum() + 1e3 * vT.sum()), (r0, v0, bc))
        return [x.detach().cpu().numpy() for x in (rT, vT, *g)]

    for a, b in zip(run(pop), run(_take(pop, EDGE))):
        assert np.array_equal(a[:EDGE], b)


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT, la.SPLIT_ALL32])
@pytest.mark.parametrize("n", [70, EDGE + 70])
def test_no_force_where_none_is_asked_for(precision, n):
    """Without components an object moves along its velocity, also at the origin and infinitely far,
    where the powers of the radius are not finite."""
    r = np.zeros((n, 3))
    r[:, 0] = np.arange(n)
    r[3] = [np.inf, 0.0, 0.0]
    r[5] = [0.0, 1.0e300, -1.0e-200]
    v = np.zeros_like(r)
    v[:, 2] = np.arange(n) * 1.0e-3
    with la.Engine(la.EngineConfig(precision=precision, components=0, cutoff_km=10.0, dt=1.0)) as eng:
        eng.set_objects(rx=r[:, 0], ry=r[:, 1], rz=r[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2], radius_m=np.ones(n))
        eng.propagate(3)
        r1, v1 = eng.state()
    assert np.array_equal(v1, v)
    np.testing.assert_array_equal(r1[:, :2], r[:, :2])
    np.testing.assert_allclose(r1[:, 2], r[:, 2] + 3.0 * v[:, 2], rtol=1e-14, atol=1e-14)
