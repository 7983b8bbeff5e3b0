"""The device minimiser's recursion against the host's search at its edges: no
correction pair, a ring of pairs not yet full, full and wrapped; and vectors
long enough that a reduction's blocks stride over them."""
import numpy as np
import pytest

from mdcore import native, synthetic
from mdcore.engine import HipEngine, RunOptions, minimise
from mdcore.system import HarmonicBondForce, OpenMMSystem

pytestmark = pytest.mark.gpu


# molecules of the solute, waters, iterations a round
@pytest.mark.parametrize("residues, waters, iterations", [(0, 700, 1), (0, 700, 2), (40, 700, 7), (0, 700, 9), (0, 29500, 2)])
def test_search_follows_the_host(residues, waters, iterations):
    b = synthetic.build(residues, waters, 0, "cube", 8)
    host = HipEngine(b.system, b.state, RunOptions())
    dev = HipEngine(b.system, b.state, RunOptions())
    start, _ = host.potential()
    h = minimise(host, iterations, 10.0)
    d = dev._native.minimise(iterations, 10.0)
    host.destroy()
    dev.destroy()
    print(start, h.energy, d["energy"])
    # only the order of sums differs (1e-16 of a product), which a few iterations
    # carry into the fixed-point coordinates' last bits: well below 1e-6
    assert abs(d["energy"] - h.energy) < 1e-6 * abs(h.energy) + 1e-3
    assert d["energy"] < start


def test_a_search_cut_short_leaves_nothing_behind():
    """An evaluation that fails just after its trial point left the fixed-point
    range: the next minimisation, of ordinary positions, knows nothing of it."""
    bond = HarmonicBondForce(np.array([0], np.int32), np.array([1], np.int32), np.array([0.4]), np.array([1e4]))
    s = native.NativeSystem(OpenMMSystem(((3, 0, 0), (0, 3, 0), (0, 0, 3)), np.array([12.0, 12.0]),
                                         np.zeros(0, np.int32), np.zeros(0, np.int32), np.zeros(0), [bond]))
    limit = 2147483648.0
    s.set_positions([limit - 0.3, 0.0, 0.0, limit - 1e-4, 0.0, 0.0])
    with pytest.raises(native.MdError, match="fixed-point range"):
        s.minimise(5, 1e-3)  # the first trial moves the second atom past the limit
    s.set_positions([limit - 0.3, 0.0, 0.0, limit - 1e-4, 0.0, 0.0])
    s.inject_fault(1)  # the starting point's evaluation passes, that trial's does not
    with pytest.raises(native.MdError, match="fault injected"):
        s.minimise(5, 1e-3)
    s.inject_fault(-1)
    s.set_positions([0.0, 0.0, 0.0, 0.3, 0.0, 0.0])
    done = s.minimise(20, 1e-3)
    s.close()
    assert done["energy"] < 1e-6
