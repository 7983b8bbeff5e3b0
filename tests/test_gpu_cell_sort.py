"""The cell sort as one workgroup per replica and as separate passes give the
same order: a replica alone takes the first up to 12,288 atoms and the second
past that, a batch takes the second when any of its replicas is larger.
Trajectories through rebuilds are bit-identical either way."""
import numpy as np
import pytest

from mdcore import synthetic
from mdcore.engine import HipBatch, HipEngine, RunOptions

pytestmark = pytest.mark.gpu


def _engine(b):
    e = HipEngine(b.system, b.state, RunOptions(timeStep=0.0005, friction=10.0, seed=4))
    e.minimise(20, 100.0)
    e.setVelocitiesToTemperature(300.0, 4)
    return e


@pytest.mark.parametrize("waters,shape", [(350, "cube"), (427, "octahedron"), (4095, "cube"), (4096, "cube")])
def test_sorted_alone_equals_sorted_beside_a_larger_replica(waters, shape):
    small = synthetic.build(0, waters, 0, shape, 7)
    large = synthetic.build(0, 4097, 0, "cube", 8)
    assert large.system.particleCount == 12291
    alone, beside, other = _engine(small), _engine(small), _engine(large)
    batch = HipBatch([beside, other])
    alone.run(60)
    batch.run(60)
    assert alone.verletFlags()["rebuilds"] > 2
    assert np.array_equal(alone.positions(), beside.positions())
    assert np.array_equal(alone.velocities(), beside.velocities())
    batch.destroy()
    for e in (alone, beside, other):
        e.destroy()
