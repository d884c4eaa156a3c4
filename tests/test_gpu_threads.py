"""Handles of their own in several host threads at once: creation, runs whose graphs are captured anew, gradients,
read-backs and the seam-wrap call give what each gives alone."""
import threading

import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu


def job(T, m, i, out):
    g = np.random.default_rng(i)
    R, n = int(g.choice([1, 3])), int(g.integers(20, 1500))
    res = []
    for mode in (1, 2, 1):
        b = T.Batch(m, [n] * R, [T.params(**P.PHYS, sigma=0.05)] * R)
        b.set_mode(mode)
        b.init_random(np.arange(R, dtype=np.uint64) + i)
        b.stage_noise(g.normal(0, 0.1, (10, n * R)).astype(np.float32))
        for _ in range(6):
            assert b.run(int(g.integers(1, 10)), 0) == T.OK  # another graph for another number of steps
            s, o = b.get_state(), b.get_outputs()
            res += [s.x, s.vid, o.r3d, o.nbr]
        if mode == 1:
            res += list(b.adjoint(4, T.loss(0.8, 1.0, 0.1, T.target_field(4)), 0, 2)[2:])
            b.set_launch(4, 64)
            assert b.run(2, 0) == T.OK
            res.append(b.get_state().theta)
        b.close()
    a = g.random((200, 2))
    res += list(T.seam_wrap(a, a + g.normal(0, 5, (200, 2)), 4)[1:])
    out[i] = res


def test_threads_with_their_own_handles(T):
    m, _ = P.mesh_and_tables(32, 0.05)
    alone, together, failed = {}, {}, []

    def guarded(i):
        try:
            job(T, m, i, together)
        except BaseException as e:  # noqa: BLE001 (reported below)
            failed.append((i, repr(e)))

    for i in range(8):
        job(T, m, i, alone)
    for _ in range(3):
        together.clear()
        threads = [threading.Thread(target=guarded, args=(i,)) for i in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not failed, failed
        for i in alone:
            assert all(np.array_equal(a, b) for a, b in zip(alone[i], together[i])), i
