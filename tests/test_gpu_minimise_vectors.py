"""The device minimiser's recursion against the host's search at its edges: no
correction pair, a ring of pairs not yet full, full and wrapped; and vectors
long enough that a reduction's blocks stride over them."""
import pytest

from mdcore import synthetic
from mdcore.engine import HipEngine, RunOptions, minimise

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
