"""Gradients of loss weights far up the FP32 range: the reverse pass is linear in the weights, so weights times
2^e give gradients times 2^e, exactly, as long as an adjoint and one step's growth of it fit in FP32. Every form
of the reverse pass (engine_adjoint.cpp) holds that range: the whole tape with every state's buckets and with
the ring of buckets, and the checkpointed segments."""
import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu

KEYS = ("d_v0", "d_mu", "d_k", "d_tau", "loss_order", "loss_velocity")


def gradients(T, m, form, n, k, w_order, w_velocity, monkeypatch, steps=8):
    monkeypatch.delenv("TISSUE_ADJOINT_BUCKET_KB", raising=False)
    if form == "ring":  # the tape and a little more than eight bucket sets
        sets_kb = 8 * (m.info()["nv"] * 37 + n * 16 + 8192) // 1024
        monkeypatch.setenv("TISSUE_ADJOINT_BUCKET_KB", str((steps + 1) * n * 44 // 1024 + 1 + sets_kb))
    sim = T.Sim(m, T.params(**dict(P.PHYS, k=k), sigma=0.1), n)
    sim.set_mode(T.MODE_STEP_KERNEL)
    if form == "segments":
        sim.set_visit_check()
    sim.init_random(0)
    sim.stage_noise(T.gen_noise(2, 0.1, steps, n))
    code, g, dth, dx, dy = sim.adjoint(steps, T.loss(0.8, w_order, w_velocity, T.target_field(4)), 0, 4)
    assert code == T.OK
    sim.close()
    return np.concatenate([[g[q] for q in KEYS], dth, dx, dy])


@pytest.mark.parametrize("form", ["whole", "ring", "segments"])
@pytest.mark.parametrize("w,n,k,exponents", [((1.0, 0.0), 400, 1000.0, (60, 100, 126)), ((0.0, 1.0), 100, 10.0, (60, 110)),
                                             ((0.0, 1.0), 400, 10.0, (112,)), ((0.0, 1.0), 400, 1000.0, (60, 92, 100))])
def test_gradients_scale_with_the_weights(T, monkeypatch, form, w, n, k, exponents):
    m, _ = P.mesh_and_tables(22, 0.1)
    base = gradients(T, m, form, n, k, *w, monkeypatch)
    assert np.isfinite(base).all() and np.abs(base).max() > 0
    for e in exponents:
        got = gradients(T, m, form, n, k, w[0] * 2.0**e, w[1] * 2.0**e, monkeypatch)
        assert np.isfinite(got).all(), e
        assert np.array_equal(got, base * 2.0**e), e
