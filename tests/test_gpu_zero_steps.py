"""A call of no steps, with and without noise rows: OK, and state, outputs and order history as they were (the
empty remainder of a run in chunks)."""
import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("n", [1, 100])
def test_no_steps(T, n, mode):
    m, _ = P.mesh_and_tables(22, 0.1)
    sim = T.Sim(m, T.params(**P.PHYS, sigma=0.1), n)
    sim.set_mode(mode)
    empty = np.zeros((0, n), np.float32)
    with pytest.raises(T.TissueError) as e:  # no state yet
        sim.step(0, empty)
    assert e.value.code == T.E_INVALID_ARG
    sim.init_random(1)
    for before in (0, 2):
        assert sim.step(before, T.gen_noise(3, 0.1, before, n)) == T.OK
        s, o, h = sim.get_state(), sim.get_outputs(), sim.order()
        assert sim.step(0, empty) == T.OK
        assert sim.step(0) == T.OK
        t, q, g = sim.get_state(), sim.get_outputs(), sim.order()
        assert all(np.array_equal(getattr(s, k), getattr(t, k)) for k in ("x", "y", "theta", "vid"))
        assert all(np.array_equal(getattr(o, k), getattr(q, k)) for k in ("vx", "vy", "r3d", "face", "nbr"))
        assert all(np.array_equal(a, b) for a, b in zip(h, g)) and len(g[0]) == before
    sim.close()
