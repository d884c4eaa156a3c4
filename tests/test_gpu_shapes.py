"""Launch shapes that read the buckets' occupancy masks and shapes whose steps do not keep them, taken
in turn by one simulation: each stretch equals a fresh simulation started from the same state at the
same shape, bit for bit (the masks are made anew when a shape that reads them follows one that does
not)."""
import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu

# (lanes, block) on the 10,337-vertex mesh (324 mask words): 8 words per particle of the tile at most
KEEPS, LACKS = (2, 256), (32, 64)


@pytest.mark.parametrize("order", [(KEEPS, LACKS, KEEPS), (LACKS, KEEPS, LACKS, KEEPS)])
@pytest.mark.parametrize("n", [33, 2000])
def test_shapes_in_turn(T, n, order):
    m, _ = P.mesh_and_tables(32, 0.05)
    prm = T.params(**P.PHYS, sigma=0.05)
    noise = T.gen_noise(7, 0.1, 4, n)
    sim = T.Sim(m, prm, n)
    sim.set_mode(T.MODE_STEP_KERNEL)
    sim.init_random(3)
    for shape in order:
        sim.set_launch(*shape)
        s = sim.get_state()
        ref = T.Sim(m, prm, n)
        ref.set_mode(T.MODE_STEP_KERNEL)
        ref.set_launch(*shape)
        ref.set_state(s.x, s.y, s.theta, s.vid)
        assert sim.step(4, noise) == T.OK and ref.step(4, noise) == T.OK
        a, b = sim.get_state(), ref.get_state()
        for k in ("x", "y", "theta", "vid"):
            assert np.array_equal(getattr(a, k), getattr(b, k)), (shape, k)
        assert np.array_equal(sim.get_outputs().nbr, ref.get_outputs().nbr), shape
        ref.close()
    sim.close()
