"""A step's mesh and bonded terms beside its list and pairs: the same bits as in
one line.  Steps replayed from a graph and launched one by one fork, profiled
steps do not; systems without bonded terms and batches included."""
import numpy as np
import pytest

from mdcore import synthetic
from mdcore.engine import HipBatch, HipEngine, RunOptions

pytestmark = pytest.mark.gpu


def _engine(residues, waters, seed=5):
    b = synthetic.build(residues, waters, 0, "cube", 19)
    return HipEngine(b.system, b.state, RunOptions(timeStep=0.0005, friction=10.0, seed=seed))


def _same(a, b):
    assert np.array_equal(a.positions(), b.positions())
    assert np.array_equal(a.velocities(), b.velocities())


@pytest.mark.parametrize("residues, waters", [(0, 700), (40, 700), (0, 9000)])
def test_forked_steps_equal_steps_in_a_line(residues, waters):
    graph, single, line = (_engine(residues, waters) for _ in range(3))
    for _ in range(3):  # replays of the same graph, with eager work between them
        graph.run(8)
        energy, forces = graph.potential()
        for _ in range(8):
            single.run(1)
        line.profileStep(8)
        _same(graph, single)
        _same(graph, line)
        e2, f2 = single.potential()
        assert e2 == energy and np.array_equal(f2, forces)
    for e in (graph, single, line):
        e.destroy()


def test_forked_batch_equals_a_batch_in_a_line():
    sizes = [(40, 700), (0, 900), (0, 1400)]
    forked, line = ([_engine(r, w, k) for k, (r, w) in enumerate(sizes)] for _ in range(2))
    a, b = HipBatch(forked), HipBatch(line)
    a.run(12)
    b.profileStep(12)
    for x, y in zip(forked, line):
        _same(x, y)
    a.destroy()
    b.destroy()
    for e in forked + line:
        e.destroy()
