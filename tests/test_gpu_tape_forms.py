"""The whole tape's two forms (engine_adjoint.cpp) really taken, and their gradients those of the checkpointed
form bit for bit: memory budgets that hold the tape and exactly eight bucket sets (the ring), or every state's.
The device memory that the calls leave held tells the forms apart: all else is the same in both, so they differ
by their sets, to the 2 MiB blocks in which each call's memory is given out. Horizons on either side of half a ring, of the
ring and of its second turn; replicas sparse on their mesh (a refilled set is cleared where its old state
was) and dense (cleared whole); raw buckets and sorted ones (the finalize pass on the side stream)."""
import ctypes as C

import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu

# mesh frequency, sigma, sizes; 64 replicas, so that a bucket set is 24 and 12 MB
SPARSE = (32, 0.05, [60, 1, 77, 250] * 16)
DENSE = (22, 0.1, [700, 650, 610, 33 + 650] * 16)


def free_bytes(T):
    T.lib()  # the library first: its HIP runtime is the one opened here (by soname)
    rt = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert rt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("sorted_buckets", [False, True])
@pytest.mark.parametrize("system", [SPARSE, DENSE], ids=["sparse", "dense"])
@pytest.mark.parametrize("steps", [7, 8, 9, 12, 13, 19])
def test_forms_are_taken_and_agree(T, monkeypatch, steps, system, sorted_buckets):
    freq, sigma, sizes = system
    m, _ = P.mesh_and_tables(freq, sigma)
    nv, R, n = m.info()["nv"], len(sizes), sum(sizes)
    assert (8 * n >= R * nv) == (system is DENSE)
    if sorted_buckets:
        monkeypatch.setenv("TISSUE_SORTED_BUCKETS", "1")
    else:
        assert 2 * max(sizes) <= nv
    loss = T.loss(0.8, 1.0, 0.1, T.target_field(4))
    start = [m.random_init_host(60 + r, k) for r, k in enumerate(sizes)]
    x, y, th = (np.concatenate([s[q] for s in start]) for q in range(3))
    noise = np.random.default_rng(2).normal(0, 0.1, (steps, n)).astype(np.float32)
    tape = (steps + 1) * n * 24 + steps * n * 20
    set_bytes = R * nv * 36 + n * 16 + R * 8 + R * 4 * ((nv + 31) // 32) + 4096
    first, held = None, {}
    for form, sets in (("anew", None), ("ring", 8), ("kept", steps + 2)):
        budget = 0 if sets is None else -(-(tape + sets * set_bytes) // 1024)
        monkeypatch.setenv("TISSUE_ADJOINT_BUCKET_KB", str(budget))
        b = T.Batch(m, sizes, [T.params(**dict(P.PHYS, tau=0.5 + r % 4), sigma=sigma) for r in range(R)])
        b.set_mode(T.MODE_STEP_KERNEL)
        b.stage_noise(noise)
        b.set_state(x, y, th)
        assert b.run(1, 0) == T.OK  # what every run holds
        before = free_bytes(T)
        for call in range(2):  # the second on sets that the first one filled
            b.set_state(x, y, th)
            code, g, dth, dx, dy = b.adjoint(steps, loss, 0, 4)
            assert code == T.OK
            out = [dth, dx, dy] + [np.array([q[k] for q in g]) for k in ("loss", "phi_final", "d_tau", "d_mu", "d_v0", "d_k")]
            first = first or out
            for a, c in zip(first, out):
                assert np.array_equal(a, c), (form, call)
        held[form] = before - free_bytes(T)
        b.close()
    assert abs(held["kept"] - held["ring"] - (steps + 2 - 8) * set_bytes) <= 2**22 < set_bytes / 2, (held, set_bytes)
