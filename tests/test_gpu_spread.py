"""Charge spreading at the forms its tiles take: one super-cluster to a
workgroup and two (from 1,024 super-clusters in the launch), a last workgroup
with one, stencil boxes that exceed the tile (sparse atoms on a fine mesh),
meshes that a box wraps more than once, and super-clusters without charge,
alone and as either one of a pair.
Against the oracle on the same mesh."""
import copy

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


TILE = 5632  # points of a spreading tile


def _slabs(b, period, phase):
    """The system with the charges of whole waters cleared in slabs normal to x."""
    system = copy.deepcopy(b.system)
    nb = system.force("NonbondedForce")
    oxygen = np.asarray(b.state.positions).reshape(-1, 3)[::3]
    off = np.floor(oxygen[:, 0] / period + phase).astype(int) % 2 == 0
    nb.charge = np.where(np.repeat(off, 3), 0.0, nb.charge)
    return system


def _pairs(system, x, mesh):
    """How many pairs of super-clusters have charge in one only, the (first,
    second) one, with a stencil box past the tile there: the cell sort of a cube
    with its cells' walk, as the engine lays out slots."""
    L = system.boxVectors[0][0]
    f = np.asarray(x).reshape(-1, 3) / L
    f -= np.floor(f)
    g = max(2, 2 * int(L / 0.6))
    rank = np.empty(g ** 3, int)
    rank[native.probe_cell_order((g, g, g))] = np.arange(g ** 3)
    c = np.minimum((f * g).astype(int), g - 1)
    order = np.argsort(rank[(c[:, 0] * g + c[:, 1]) * g + c[:, 2]], kind="stable")
    q = system.force("NonbondedForce").charge[order]
    cell = np.floor(f[order] * mesh)
    found = [0, 0]
    for S in range(0, -(-len(q) // 64) - 1, 2):
        part = [slice(64 * S, 64 * S + 64), slice(64 * S + 64, 64 * S + 128)]
        live = [np.any(q[p] != 0.0) for p in part]
        if live[0] == live[1]:
            continue
        k = 0 if live[0] else 1
        at = cell[part[k]][q[part[k]] != 0.0]
        found[k] += np.prod(at.max(axis=0) - at.min(axis=0) + 5) > TILE
    return found


def test_paired_super_clusters_one_without_charge():
    """A pair of which one has no charge and the other a stencil box past the
    tile: the batch, which pairs, against each replica alone, which does not."""
    b = synthetic.build(0, 662, 0, "cube", 15)
    systems = [_slabs(b, period, phase) for period, phase in [(0.9, 0.0), (0.9, 0.4), (1.0, 0.6), (1.1, 0.8)]]
    x, mesh = b.state.positions, 72
    found = np.sum([_pairs(s, x, mesh) for s in systems], axis=0)
    print("pairs with charge in the first only, the second only:", found)
    assert found.min() > 0
    opts = RunOptions(timeStep=0.0005, friction=10.0, seed=1, mesh=(mesh,) * 3)
    alone = [HipEngine(s, b.state, opts) for s in systems]
    many = [HipEngine(s, b.state, opts) for s in systems * 9]
    assert sum(-(-e.particleCount // 64) for e in many) >= 1024
    batch = HipBatch(many)
    batch.run(4)
    for e in alone:
        e.run(4)
    for k, e in enumerate(many):
        assert np.array_equal(e.positions(), alone[k % 4].positions()), k
        assert np.array_equal(e.velocities(), alone[k % 4].velocities()), k
    batch.destroy()
    for e in alone + many:
        e.destroy()
    _check(systems[0], x, (mesh,) * 3)
