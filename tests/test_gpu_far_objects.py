"""Objects so far away that the square of their distance overflows: the forces there are 0 and the
objects move on along their velocity, in the engine and in the differentiable propagation."""
import numpy as np
import pytest
import torch

import ladds_amd as la
from ladds_amd import adjoint

pytestmark = pytest.mark.gpu

FAR = np.array([[1.0e160, -3.0e158, 2.0e157], [-2.0e200, 5.0, 0.0], [0.0, 7.0e154, 1.0e155]])


def _population(n):
    """Objects in low orbits with the far ones among them."""
    pop = la.generate_population(0, 0x1ADD5 + 81, n)
    at = np.array([2, n // 2, n - 1])
    pop.rx[at], pop.ry[at], pop.rz[at] = FAR.T
    return pop, at


@pytest.mark.parametrize("precision", [la.FP64, la.SPLIT, la.SPLIT_ALL32])
@pytest.mark.parametrize("n", [70, 262144 + 70])  # staged environments or not
def test_kepler_alone(precision, n):
    pop, at = _population(n)
    with la.Engine(la.EngineConfig(precision=precision, components=la.KEP, cutoff_km=10.0, dt=10.0)) as eng:
        eng.set_objects(pop)
        eng.propagate(3)
        r, v = eng.state()
    assert np.isfinite(r).all() and np.isfinite(v).all()
    assert np.array_equal(v[at], pop.v()[at])
    np.testing.assert_allclose(r[at], FAR + 30.0 * pop.v()[at], rtol=1e-14)


@pytest.mark.parametrize("mask", [la.SOL, la.LUN, la.KEP | la.SOL | la.LUN])
def test_third_bodies(mask):
    """The third bodies' direct terms vanish as well; what is left does not depend on the place."""
    pop, at = _population(70)
    with la.Engine(la.EngineConfig(components=mask, cutoff_km=10.0, dt=10.0)) as eng:
        eng.set_objects(pop)
        eng.propagate(3)
        r, v = eng.state()
    assert np.isfinite(r).all() and np.isfinite(v).all()
    kick = v[at] - pop.v()[at]
    assert np.abs(kick).max() < 1.0
    np.testing.assert_allclose(kick - kick[0], 0.0, atol=1e-13)


def test_gradient():
    pop, at = _population(70)
    t = lambda x: torch.tensor(np.ascontiguousarray(x), dtype=torch.float64, device="cuda:0")
    plan = adjoint.AdjointPlan(pop.n, 5, 10.0, components=la.KEP, checkpoint_every=2)
    r0, v0, bc = (t(x).requires_grad_() for x in (pop.r(), pop.v(), pop.bc_inv))
    rT, vT = adjoint.propagate(r0, v0, bc, plan, aom=t(pop.aom), cr=t(pop.cr))
    g_r, g_v = (g.cpu().numpy() for g in torch.autograd.grad(rT.sum() + 3.0 * vT.sum(), (r0, v0)))
    plan.close()
    assert np.array_equal(vT.detach().cpu().numpy()[at], pop.v()[at])
    assert np.isfinite(g_r).all() and np.isfinite(g_v).all()
    # rT = r0 + 50 s v0, vT = v0
    np.testing.assert_allclose(g_r[at], 1.0, rtol=1e-14)
    np.testing.assert_allclose(g_v[at], 53.0, rtol=1e-14)
