"""Calls that ask for terabytes of device memory are refused, and leave nothing behind: the next, ordinary call
allocates again and gives what an engine that never saw the refused one gives."""
import ctypes as C

import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu
N, HUGE = 1000, 2**31 - 1  # 8.6e12 bytes of noise rows


def refused(T, code):
    assert code == T.E_HIP
    assert b"memory" in T.lib().tissue_error_string()


def test_call_noise(T):
    m, _ = P.mesh_and_tables(22, 0.1)
    noise = T.gen_noise(5, 0.1, 4, N)

    def run(refuse):
        sim = T.Sim(m, T.params(**P.PHYS, sigma=0.1), N)
        sim.init_random(1)
        assert sim.step(3, noise[:3]) == T.OK
        if refuse:
            refused(T, T.lib().tissue_step(sim.h, HUGE, noise.ctypes.data_as(C.POINTER(C.c_float))))
        assert sim.step(2, noise[2:]) == T.OK
        return sim

    same_state(run(True), run(False))


def test_staged_noise(T):
    m, _ = P.mesh_and_tables(22, 0.1)
    noise = T.gen_noise(6, 0.1, 4, N)

    def run(refuse):
        sim = T.Sim(m, T.params(**P.PHYS, sigma=0.1), N)
        sim.init_random(1)
        sim.stage_noise(noise)
        if refuse:
            refused(T, T.lib().tissue_stage_noise(sim.h, noise.ctypes.data_as(C.POINTER(C.c_float)), HUGE))
            with pytest.raises(T.TissueError):  # the rows went with their buffer
                sim.step_staged(1, 0)
        sim.stage_noise(noise[:3])
        assert sim.step_staged(3, 0) == T.OK
        return sim

    same_state(run(True), run(False))


def test_order_partials(T):
    m, _ = P.mesh_and_tables(22, 0.1)
    start = m.random_init_host(3, N)

    def run(refuse):
        b = T.Batch(m, [N], [T.params(**P.PHYS, sigma=0.1)])
        b.set_mode(T.MODE_STEP_KERNEL)
        b.set_state(*start[:3])
        assert b.run(2) == T.OK
        if refuse:
            b.set_launch(0, 0, HUGE)
            with pytest.raises(T.TissueError) as e:
                b.run(1)
            refused(T, e.value.code)
            b.set_launch()
        assert b.run(2) == T.OK
        return b

    same_state(run(True), run(False))


def test_checkpoints(T, monkeypatch):
    monkeypatch.setenv("TISSUE_ADJOINT_BUCKET_KB", "0")  # segments
    m, _ = P.mesh_and_tables(22, 0.1)
    loss = T.loss(0.8, 1.0, 0.1, T.target_field(4))

    def run(refuse):
        sim = T.Sim(m, T.params(**P.PHYS, sigma=0.1), N)
        sim.set_mode(T.MODE_STEP_KERNEL)
        sim.init_random(1)
        assert sim.adjoint(8, loss, -1, 4)[0] == T.OK
        if refuse:
            with pytest.raises(T.TissueError) as e:
                sim.adjoint(2**30, loss, -1, 1)  # a checkpoint a step: 2^30 states
            refused(T, e.value.code)
        out = sim.adjoint(4, loss, -1, 4)
        assert out[0] == T.OK
        return sim, out

    (a, ga), (b, gb) = run(True), run(False)
    assert all(np.array_equal(p, q) for p, q in zip(ga[2:], gb[2:]))
    same_state(a, b)


def same_state(a, b):
    s, t = a.get_state(), b.get_state()
    assert all(np.array_equal(getattr(s, k), getattr(t, k)) for k in ("x", "y", "theta", "vid"))
    a.close(), b.close()
