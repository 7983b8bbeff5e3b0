"""The cluster integrator's forms: clusters of one heavy atom and its
hydrogens take a kernel with the constraints' atoms fixed, all others the
general one.  Naming a constraint's atoms the other way round changes no sign
that survives, so it gives the same bits; constraints in another order, or a
hydrogen before its heavy atom, take the general kernel, whose sums run in
that order, and agree to the constraint tolerance."""
import numpy as np
import pytest

from mdcore import synthetic
from mdcore.engine import HipEngine, RunOptions

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def start():
    b = synthetic.build(200, 480, 2, "cube", 21)
    e = HipEngine(b.system, b.state, RunOptions(timeStep=0.0005, friction=10.0, seed=2))
    e.minimise(100, 10.0)
    e.setVelocitiesToTemperature(300.0, 2)
    e.run(40)
    out = b.system, b.state.boxVectors, e.positions(), e.velocities()
    e.destroy()
    return out


def _run(system, box, x, v, integrator, steps):
    from mdcore.state import OpenMMState
    e = HipEngine(system, OpenMMState(box, x, v), RunOptions(timeStep=0.001, seed=9, integrator=integrator))
    e.run(steps)
    out = e.positions().reshape(-1, 3), e.velocities().reshape(-1, 3)
    e.destroy()
    return out


@pytest.mark.parametrize("integrator", ["LangevinMiddle", "Verlet"])
def test_constraint_direction_changes_no_bit(start, integrator):
    system, box, x, v = start
    p1, p2 = system.constraintP1.copy(), system.constraintP2.copy()
    straight = _run(system, box, x, v, integrator, 20)
    flip = np.arange(len(p1)) % 3 != 0
    system.constraintP1, system.constraintP2 = np.where(flip, p2, p1), np.where(flip, p1, p2)
    flipped = _run(system, box, x, v, integrator, 20)
    system.constraintP1, system.constraintP2 = p1, p2
    for a, b in zip(straight, flipped):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("integrator", ["LangevinMiddle", "Verlet"])
def test_constraint_order_stays_within_the_tolerance(start, integrator):
    system, box, x, v = start
    keep = system.constraintP1, system.constraintP2, system.constraintDistance
    straight = _run(system, box, x, v, integrator, 3)
    system.constraintP1, system.constraintP2, system.constraintDistance = (a[::-1].copy() for a in keep)
    reversed_ = _run(system, box, x, v, integrator, 3)
    d = np.linalg.norm(reversed_[0][keep[0]] - reversed_[0][keep[1]], axis=1)
    system.constraintP1, system.constraintP2, system.constraintDistance = keep
    # each path's SHAKE stops within 1e-6 of the length (0.15 nm at most): the
    # paths may differ by twice that a step, and a step's difference is carried
    # on as velocity by the next two
    assert np.max(np.abs(straight[0] - reversed_[0])) < 3 * (1 + 2 + 3) * 2e-6 * 0.15
    assert np.max(np.abs(d / keep[2] - 1)) < 2e-6
