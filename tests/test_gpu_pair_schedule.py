"""How the pair kernel's list is shared out among its waves never shows in the
results: every wave count and segment length gives the same forces, bit for
bit, on lists with fewer segments than waves, runs that start and end inside
a super-cluster, and counts that the 8 XCD ranges do not divide."""
import numpy as np
import pytest

from mdcore import native, synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def system():
    b = synthetic.build(60, 500, 2, "octahedron", 11)
    s = native.NativeSystem(b.system)
    s.set_positions(b.state.positions)
    total, groups, forces = s.evaluate()
    yield s, b.state.positions, total, groups, forces
    s.close()


@pytest.mark.parametrize("entries,waves", [(8, 1), (8, 7), (8, 8), (8, 9), (8, 100), (8, 100000), (16, 333),
                                           (64, 64), (256, 5), (256, 4096)])
def test_any_schedule_gives_the_same_forces(system, entries, waves):
    s, x, total, groups, forces = system
    s.set_pair_schedule(entries, waves, False)
    s.set_positions(x)
    t, g, f = s.evaluate()
    assert t == total and np.array_equal(g, groups)
    assert np.array_equal(f, forces)
