"""How the pair kernel's list is shared out among its waves never shows in the
results: every wave count and segment length gives the same forces, bit for
bit, on lists with fewer segments than waves, runs that start and end inside
a super-cluster, and counts that the 8 XCD ranges do not divide.  An evaluation
launches the kernel with energies; steps launch the one without and the
compacted one, alone and over replicas of unequal lists."""
import numpy as np
import pytest

from mdcore import native, synthetic
from mdcore.engine import HipBatch, HipEngine, RunOptions

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


SCHEDULES = [(8, 1), (8, 7), (8, 9), (8, 100), (8, 100000), (16, 333), (64, 64), (256, 5), (256, 4096)]


def _engines(sizes):
    built = [synthetic.build(r, w, 0, shape, 12 + k) for k, (r, w, shape) in enumerate(sizes)]
    return [HipEngine(b.system, b.state, RunOptions(timeStep=0.0005, friction=10.0, seed=6)) for b in built]


def _run(sizes, entries, waves, compact):
    """Positions and velocities after a few steps, the first of which rebuilds: one system, or
    a batch of several.  The schedule is set in any case, since one tuned
    earlier in the process may be the default."""
    engines = _engines(sizes)
    batch = HipBatch(engines) if len(engines) > 1 else None
    (batch or engines[0])._native.set_pair_schedule(entries, waves, compact)
    (batch or engines[0]).run(12)
    out = [a for e in engines for a in (e.positions(), e.velocities())]
    if batch:
        batch.destroy()
    for e in engines:
        e.destroy()
    return out


@pytest.fixture(scope="module", params=["alone", "batch"])
def steps(request):
    sizes = [(60, 500, "octahedron")] if request.param == "alone" else [(0, 350, "cube"), (40, 900, "octahedron"),
                                                                        (0, 427, "cube")]
    return sizes, _run(sizes, 8, 4096, False)


@pytest.mark.parametrize("compact", [False, True])
@pytest.mark.parametrize("entries,waves", SCHEDULES)
def test_any_schedule_gives_the_same_steps(steps, entries, waves, compact):
    sizes, want = steps
    for a, b in zip(_run(sizes, entries, waves, compact), want):
        assert np.array_equal(a, b)
