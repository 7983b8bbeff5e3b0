"""The list search at the forms it takes: 16, 8 and 4 waves to a super-cluster
(by the launch's size), candidates with more images within reach than are kept
from the counting pass (small cells), an evaluation's rebuild sorted in separate
passes and a step's in one workgroup.  The list's order is the same in all, so
forces and trajectories are too; and it is complete, so forces are the
oracle's."""
import numpy as np
import pytest

import edge
import oracle as O
from mdcore import native, synthetic
from mdcore.engine import HipBatch, HipEngine, RunOptions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters, shape", [(350, "cube"), (427, "octahedron"), (1400, "octahedron"), (4000, "cube")])
def test_forces_are_the_oracles(waters, shape):
    b = synthetic.build(0, waters, 0, shape, 17)
    o = O.OracleSystem(b.system)
    s = native.NativeSystem(b.system, mesh=(32, 32, 32))
    s.set_positions(b.state.positions)
    _, _, f = s.evaluate()
    _, _, of = o.potential(b.state.positions, b.system.boxVectors, grid=(32, 32, 32))
    err, _ = edge.rel_rms_edge(f, of, b.system, b.state.positions, b.system.boxVectors, o.alpha())
    s.close()
    assert err < 2e-6, err  # the parity gate's tolerance


# 192 super-clusters alone: 16 waves; twice that: 8; six times: 4.  From 4,096
# atoms an evaluation's rebuild takes the separate passes.
@pytest.mark.parametrize("waters, copies", [(4000, 2), (4000, 6), (1365, 9), (1366, 9)])
def test_waves_and_sort_change_no_bit(waters, copies):
    b = synthetic.build(0, waters, 0, "cube", 18)
    opts = RunOptions(timeStep=0.0005, friction=10.0, seed=3)
    alone, evaluated = HipEngine(b.system, b.state, opts), HipEngine(b.system, b.state, opts)
    many = [HipEngine(b.system, b.state, opts) for _ in range(copies)]
    batch = HipBatch(many)
    evaluated.potential(b.state.positions)  # its list is the evaluation's
    for e in (alone, evaluated):
        e.run(30)
    batch.run(30)
    for e in [evaluated] + many:
        assert np.array_equal(e.positions(), alone.positions())
        assert np.array_equal(e.velocities(), alone.velocities())
    batch.destroy()
    for e in [alone, evaluated] + many:
        e.destroy()
