"""The adjoint's forms (engine_adjoint.cpp) give the same gradients bit for bit: the whole tape with every
state's vertex buckets, the whole tape with buckets made again ahead of the reverse pass (sparse replicas:
cleared where the old state was, rows asked through the occupancy mask; dense ones: cleared and read whole),
recomputed segments on several tapes (what a run with the visit check on takes), and one tape that buckets
each state anew. Horizons on either side of the ring of sets and of a segment."""
import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [1, 3, 4, 5, 8, 9, 19])
@pytest.mark.parametrize("freq,sigma,sizes", [(32, 0.05, (60, 1, 77)), (22, 0.1, (900, 33)), (32, 0.05, (1000,))])
def test_adjoint_forms_agree(T, monkeypatch, freq, sigma, sizes, steps):
    m, _ = P.mesh_and_tables(freq, sigma)
    R, n = len(sizes), sum(sizes)
    Lc = T.loss(0.8, 1.0, 0.1, T.target_field(4))
    start = [m.random_init_host(60 + r, k) for r, k in enumerate(sizes)]
    x, y, th = (np.concatenate([s[q] for s in start]) for q in range(3))
    noise = np.random.default_rng(2).normal(0, 0.1, (steps, n)).astype(np.float32)
    set_kb = (R * m.info()["nv"] * 37 + n * 16 + 16384) // 1024  # a little more than one bucket set takes
    tape_kb = (steps + 1) * n * 44 // 1024 + 1
    forms = {"whole": None, "ring": tape_kb + 9 * set_kb, "segments": None, "anew": 0}
    res = {}
    for name, budget in forms.items():
        if budget is None:
            monkeypatch.delenv("TISSUE_ADJOINT_BUCKET_KB", raising=False)
        else:
            monkeypatch.setenv("TISSUE_ADJOINT_BUCKET_KB", str(budget))
        b = T.Batch(m, sizes, [T.params(**dict(P.PHYS, tau=0.5 + r), sigma=sigma) for r in range(R)])
        b.set_mode(T.MODE_STEP_KERNEL)
        if name == "segments":
            b.set_visit_check()
        b.stage_noise(noise)
        for _ in range(2):  # a second call on the same engine, its sets filled by the first
            b.set_state(x, y, th)
            code, g, dth, dx, dy = b.adjoint(steps, Lc, 0, 4)
            assert code == T.OK
            s = b.get_state()
            out = [dth, dx, dy, s.x, s.theta, s.vid] + [np.array([q[k] for q in g]) for k in
                                                       ("loss", "phi_final", "d_tau", "d_mu", "d_v0", "d_k")]
            if "whole" in res:
                for a, c in zip(res["whole"], out):
                    assert np.array_equal(a, c), name
            else:
                res["whole"] = out
        assert len(b.order(0)[0]) == 2 * steps
        b.run(2, -1)  # the engine goes on from the final state
        b.close()
