"""Read-backs of some of the arrays (null pointers for the rest): every choice gives what the full read-back
gives and writes nothing else, at sizes on either side of the limits between one copy and the packing kernel
(16 and 128 KB, of 16 bytes a particle for the positions and of 4 for the outputs) and in several pieces."""
import ctypes as C
import itertools

import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1024, 1025, 4096, 4097, 8192, 8193, 32768, 32769, 300001])
def test_choices_of_arrays(T, n):
    m, _ = P.mesh_and_tables(32, 0.05) if n < 5000 else P.sphere_and_tables(100, 0.2, 0.01)
    sim = T.Sim(m, T.params(**P.PHYS, sigma=0.05 if n < 5000 else 0.01), n)
    sim.set_mode(T.MODE_STEP_KERNEL)
    sim.init_random(7)
    assert sim.step(1, T.gen_noise(7, 0.1, 1, n)) == T.OK
    s, o = sim.get_state(), sim.get_outputs()
    for get, full in ((T.lib().tissue_get_state, [s.x, s.y, s.theta, s.vid]),
                      (T.lib().tissue_get_outputs, [o.vx, o.vy, o.r3d, o.face, o.nbr])):
        choices = list(itertools.product((False, True), repeat=len(full)))
        for want in choices if n < 100000 else choices[1:5] + choices[-1:]:
            out = [np.full_like(a, -77) for a in full]
            ptrs = [b.ctypes.data_as(C.POINTER(C.c_float if b.dtype == np.float32 else C.c_int32)) if w else None
                    for b, w in zip(out, want)]
            assert get(sim.h, *ptrs) == T.OK
            for a, b, w in zip(full, out, want):
                assert np.array_equal(b, a if w else np.full_like(a, -77)), want
    sim.close()
