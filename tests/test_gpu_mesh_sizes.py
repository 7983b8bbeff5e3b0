"""The mesh transforms at every kind of size: each radix, lines of a single
butterfly, odd and unequal axes, planes that fit LDS and planes that do not,
runs of kz that do not divide the half spectrum,
the longest axes.  Forces against the f64
oracle on the same mesh, at the parity gate's tolerance (2e-6 relative RMS);
reciprocal energies at 1e-5."""
import numpy as np
import pytest

import edge
import oracle as O
from mdcore import native, synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["cube", "octahedron"])
def built(request):
    b = synthetic.build(40, 480, 2, request.param, 3)
    return b, O.OracleSystem(b.system)


@pytest.mark.parametrize("mesh", [(32, 32, 32), (35, 27, 30), (24, 40, 56), (45, 28, 25), (26, 33, 22), (7, 11, 13),
                                  (13, 5, 7), (64, 64, 64), (20, 81, 98), (128, 16, 126), (30, 120, 64)])
def test_forces_match_the_oracle_on_the_same_mesh(built, mesh):
    b, o = built
    s = native.NativeSystem(b.system, mesh=mesh)
    s.set_positions(b.state.positions)
    for _ in range(2):  # the second evaluation finds the grid as the first left it
        _, g, f = s.evaluate()
        _, og, of = o.potential(b.state.positions, b.system.boxVectors, grid=mesh)
        err, _ = edge.rel_rms_edge(f, of, b.system, b.state.positions, b.system.boxVectors, o.alpha())
        assert err < 2e-6, err
        assert abs(g[4] - og[4]) <= 1e-5 * abs(og[4])
    s.close()


# Axes of more than 616 points, on which a workgroup takes fewer lines, in each
# of the three passes.  The short axes are odd (see test_gpu_spread).  A force
# from the mesh is a difference of neighbouring f32 potentials times the points
# per nm, so its rounding grows with them: four times the gate's tolerance,
# which axes of 160 points keep, at 640.
@pytest.mark.parametrize("mesh", [(9, 9, 616), (9, 9, 640), (9, 640, 9), (640, 9, 9), (11, 9, 625), (9, 637, 11),
                                  (630, 11, 13)])
def test_the_longest_axes(mesh):
    b = synthetic.build(40, 480, 2, "cube", 3)
    o = O.OracleSystem(b.system)
    s = native.NativeSystem(b.system, mesh=mesh)
    s.set_positions(b.state.positions)
    _, og, of = o.potential(b.state.positions, b.system.boxVectors, grid=mesh)
    for _ in range(2):
        _, g, f = s.evaluate()
        err, _ = edge.rel_rms_edge(f, of, b.system, b.state.positions, b.system.boxVectors, o.alpha())
        assert err < 8e-6, err
        assert abs(g[4] - og[4]) <= 1e-5 * abs(og[4])
    s.close()


@pytest.mark.parametrize("mesh", [(9, 9, 648), (648, 9, 9), (9, 1024, 9)])
def test_a_longer_axis_is_refused_by_name(mesh):
    b = synthetic.build(0, 480, 0, "cube", 3)
    with pytest.raises(native.MdError, match="at most 640"):
        native.NativeSystem(b.system, mesh=mesh)
