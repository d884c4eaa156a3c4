"""Adjoints whose horizons take turns on one engine: a short one whose run keeps every state's bucket sets and
a long one that makes them again in a ring (the memory budget lets only the short one keep them). The
gradients are a fresh engine's, and from the second turn on the engine holds the same device memory after each
call: nothing is freed and allocated anew."""
import ctypes as C

import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu


def free_bytes(T):
    T.lib()  # the library first: its HIP runtime is the one opened here (by soname)
    rt = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert rt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("horizons,sets", [((4, 40), 20), ((40, 4), 20), ((3, 60, 7), 12), ((60, 4), 400)])
def test_alternating_horizons(T, monkeypatch, horizons, sets):
    m, _ = P.mesh_and_tables(32, 0.05)
    R, n, T_max = 16, 16 * 500, max(horizons)
    set_bytes = R * m.info()["nv"] * 37 + n * 16 + 8192
    monkeypatch.setenv("TISSUE_ADJOINT_BUCKET_KB", str(((T_max + 1) * n * 44 + sets * set_bytes) // 1024))
    start = [m.random_init_host(60 + r, 500) for r in range(R)]
    x, y, th = (np.concatenate([s[q] for s in start]) for q in range(3))
    loss = T.loss(0.8, 1.0, 0.1, T.target_field(4))
    noise = np.random.default_rng(2).normal(0, 0.1, (T_max, n)).astype(np.float32)

    def engine():
        b = T.Batch(m, [500] * R, [T.params(**P.PHYS, sigma=0.05)] * R)
        b.set_mode(T.MODE_STEP_KERNEL)
        b.stage_noise(noise)
        return b

    def call(b, steps):
        b.set_state(x, y, th)
        code, _, dth, dx, dy = b.adjoint(steps, loss, 0, 4)
        assert code == T.OK
        return dth, dx, dy

    ref = {}
    for steps in horizons:
        b = engine()
        ref[steps] = call(b, steps)
        b.close()
    b, held = engine(), set()
    for turn in range(4):
        for steps in horizons:
            for a, c in zip(ref[steps], call(b, steps)):
                assert np.array_equal(a, c), (turn, steps)
            if turn > 0:
                held.add(free_bytes(T))
    assert len(held) == 1, held
    b.close()
