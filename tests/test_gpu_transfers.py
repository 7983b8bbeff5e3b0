"""Positions and velocities to the device and back: the caller's f64 rounded to
Q32.32 and to f32 as on the host, at atom counts around the padding; a refused
array leaves the state; readers in several threads do not disturb each other."""
import threading

import numpy as np
import pytest

from mdcore import native, synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[427, 448, 661])  # 1281, 1344 and 1983 atoms: 1, 0 and 63 past a multiple of 64
def system(request):
    b = synthetic.build(0, request.param, 0, "cube" if request.param != 427 else "octahedron", 3)
    s = native.NativeSystem(b.system)
    yield s, b.state.positions
    s.close()


def test_round_trip_is_the_formats_rounding(system):
    s, x = system
    rng = np.random.default_rng(5)
    x = x.reshape(-1) + rng.normal(0, 40, x.size)
    x[0], x[1], x[2] = -0.0, 2147483647.5, -2147483647.75
    x[3:5] = 2.0 ** -33, 3 * 2.0 ** -33  # ties, to even
    v = rng.normal(0, 3, x.size)
    s.set_positions(x)
    s.set_velocities(v)
    assert np.array_equal(s.positions(), np.rint(x * 2.0 ** 32) / 2.0 ** 32)
    assert np.array_equal(s.velocities(), v.astype(np.float32).astype(np.float64))


@pytest.mark.parametrize("bad", [np.nan, np.inf, 2147483648.0])
def test_refused_positions_leave_the_state(system, bad):
    s, x = system
    s.set_positions(x)
    before = s.positions()
    y = x.reshape(-1).copy()
    y[-1] = bad
    with pytest.raises(native.MdError):
        s.set_positions(y)
    w = np.zeros_like(y)
    w[-1] = np.nan
    with pytest.raises(native.MdError):
        s.set_velocities(w)
    assert np.array_equal(s.positions(), before)


def test_readers_in_threads(system):
    s, x = system
    s.set_positions(x)
    s.set_velocities(np.linspace(-1, 1, x.size))
    want, speed = s.positions(), s.velocities()
    wrong = []

    def read(get, expect):
        for _ in range(40):
            if not np.array_equal(get(), expect):
                wrong.append(get)

    threads = [threading.Thread(target=read, args=a) for a in ((s.positions, want), (s.velocities, speed)) * 2]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
