"""Charge spreading at the forms its tiles take: one super-cluster to a
workgroup and two (from 1,024 super-clusters in the launch), a last workgroup
with one, stencil boxes that exceed the tile (sparse atoms on a fine mesh),
meshes that a box wraps more than once, and super-clusters without charge.
Against the oracle on the same mesh."""
import numpy as np
import pytest

import edge
import oracle as O
from mdcore import native, synthetic
from mdcore.engine import HipBatch, HipEngine, RunOptions

pytestmark = pytest.mark.gpu


def _check(system, x, mesh, tolerance=2e-6):
    o = O.OracleSystem(system)
    s = native.NativeSystem(system, mesh=mesh)
    s.set_positions(x)
    _, _, f = s.evaluate()
    _, _, of = o.potential(x, system.boxVectors, grid=mesh)
    err, _ = edge.rel_rms_edge(f, of, system, x, system.boxVectors, o.alpha())
    s.close()
    assert err < tolerance, err


# the tiny mesh has odd axes: the Nyquist plane of an even one has two readings in
# a triclinic cell (m = n/2 and -n/2), which the oracle and the half spectrum
# take differently, and on a mesh this coarse that plane still carries weight
@pytest.mark.parametrize("mesh", [(32, 32, 32), (5, 7, 9), (96, 90, 84), (160, 150, 144)])
def test_one_system_against_the_oracle(mesh):
    b = synthetic.build(40, 480, 2, "octahedron", 13)
    _check(b.system, b.state.positions, mesh)


def test_super_clusters_without_charge():
    b = synthetic.build(0, 500, 0, "cube", 14)
    nb = b.system.force("NonbondedForce")
    nb.charge = nb.charge.copy()
    nb.charge[: nb.charge.size // 2] = 0.0
    _check(b.system, b.state.positions, (32, 32, 32))


def test_paired_super_clusters_equal_single_ones():
    """The same replica alone (one super-cluster to a workgroup) and in a batch
    of enough replicas that they pair up, odd counts included."""
    b = synthetic.build(0, 662, 0, "cube", 15)
    odd = synthetic.build(0, 683, 0, "octahedron", 16)
    systems = [b, odd] * 17
    opts = RunOptions(timeStep=0.0005, friction=10.0, seed=1)
    alone = [HipEngine(s.system, s.state, opts) for s in (b, odd)]
    many = [HipEngine(s.system, s.state, opts) for s in systems]
    assert sum(-(-e.particleCount // 64) for e in many) >= 1024
    batch = HipBatch(many)
    batch.run(6)
    for e in alone:
        e.run(6)
    for k, e in enumerate(many):
        assert np.array_equal(e.positions(), alone[k % 2].positions()), k
        assert np.array_equal(e.velocities(), alone[k % 2].velocities()), k
    batch.destroy()
    for e in alone + many:
        e.destroy()
