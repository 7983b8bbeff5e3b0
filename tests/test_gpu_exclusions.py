"""Exclusions anywhere in the list: the exclusion masks are made by looking
each excluded pair up in its super-cluster's entries, so pairs far apart in
index, pairs across a periodic boundary, atoms with many exclusions and lists
longer than one tile of 256 entries all have to find their bit.  Forces are
compared with the oracle's at the parity gate's tolerance (2e-6 relative RMS)."""
import numpy as np
import pytest

import edge
import oracle as O
from mdcore import native, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,count,skin", [("cube", 400, 0.15), ("octahedron", 400, 0.15), ("cube", 4000, 0.15),
                                              ("cube", 400, 0.5)])
def test_far_and_many_exclusions_match_the_oracle(shape, count, skin):
    b = synthetic.build(40, 620, 2, shape, 5)
    system = b.system
    x = b.state.positions.reshape(-1, 3)
    n = x.shape[0]
    rng = np.random.default_rng(count)
    nb = system.force("NonbondedForce")
    taken = set(zip(nb.exceptionP1.tolist(), nb.exceptionP2.tolist()))
    box = np.asarray(system.boxVectors)
    new = []
    while len(new) < count:
        i, j = sorted(int(v) for v in rng.integers(0, n, 2))
        d = x[j] - x[i]
        for k in (2, 1, 0):
            d = d - np.floor(d[k] / box[k, k] + 0.5) * box[k]
        # not the closest pairs: an excluded pair keeps only its Ewald term
        if i != j and (i, j) not in taken and (j, i) not in taken and 0.3 < np.linalg.norm(d) < 0.98:
            taken.add((i, j))
            new.append((i, j))
    new = np.array(new, dtype=np.int32)
    nb.exceptionP1 = np.concatenate([nb.exceptionP1, new[:, 0]])
    nb.exceptionP2 = np.concatenate([nb.exceptionP2, new[:, 1]])
    nb.exceptionChargeProd = np.concatenate([nb.exceptionChargeProd, np.zeros(count)])
    nb.exceptionSigma = np.concatenate([nb.exceptionSigma, np.ones(count)])
    nb.exceptionEpsilon = np.concatenate([nb.exceptionEpsilon, np.zeros(count)])
    o = O.OracleSystem(system)
    grid = o.default_grid(system.boxVectors)
    s = native.NativeSystem(system, mesh=grid, verlet_skin=skin)
    s.set_positions(b.state.positions)
    _, _, f = s.evaluate()
    _, _, of = o.potential(b.state.positions, system.boxVectors, grid=grid)
    err, _ = edge.rel_rms_edge(f, of, system, b.state.positions, system.boxVectors, o.alpha())
    assert err < 2e-6, err
    s.close()
