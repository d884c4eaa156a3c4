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


def _batch(T, m, sizes, raw, monkeypatch, lanes, x, y, th):
    monkeypatch.setenv("TISSUE_SORTED_BUCKETS", "0" if raw else "1")
    b = T.Batch(m, sizes, [T.params(**P.PHYS, sigma=0.1)] * len(sizes))
    monkeypatch.delenv("TISSUE_SORTED_BUCKETS")
    b.set_mode(T.MODE_STEP_KERNEL)
    b.set_launch(lanes, 256)
    b.set_visit_check()
    b.set_state(x, y, th)
    return b


@pytest.mark.parametrize("lanes", [1, 2, 4, 8])
@pytest.mark.parametrize("sizes", [(1, 2, 63), (700, 1, 65), (4000,), (4000,) * 9])
def test_walk_of_a_whole_wave(T, monkeypatch, lanes, sizes):
    """The whole-wave walk (raw buckets, and sorted ones with more lanes than the sums' layout) where its
    lists overflow (4,000 particles on 4,907 vertices: more occupied entries than the list holds, more
    pairs than a round, crowded buckets) and where waves are nearly empty, on one lane per strand and
    on several (sizes on either side of phys_lanes): raw and sorted buckets, hence two walks, give the
    same bits, and each particle's visited set is the one a plain kernel lists."""
    m, _ = P.mesh_and_tables(22, 0.1)
    n = sum(sizes)
    start = [m.random_init_host(40 + r, k) for r, k in enumerate(sizes)]
    x, y, th = (np.concatenate([s[q] for s in start]) for q in range(3))
    a, b = (_batch(T, m, sizes, raw, monkeypatch, lanes, x, y, th) for raw in (True, False))
    noise = np.random.default_rng(1).normal(0, 0.1, (2, n)).astype(np.float32)
    for q in (a, b):
        q.stage_noise(noise)
    for step in range(2):
        if n <= 4000 and len(sizes) == 1:  # the sets, listed before the step that visits them
            one = T.Sim(m, T.params(**P.PHYS, sigma=0.1), n)
            s = a.get_state()
            one.set_state(s.x, s.y, s.theta, s.vid)
            lists = one.neighbor_lists()
            one.close()
        assert a.run(1, step) == T.OK and b.run(1, step) == T.OK
        sa, sb = a.get_state(), b.get_state()
        for k in ("x", "y", "theta", "vid"):
            assert np.array_equal(getattr(sa, k), getattr(sb, k)), (step, k)
        oa, ob = a.get_outputs(), b.get_outputs()
        for k in ("vx", "vy", "r3d", "face", "nbr"):
            assert np.array_equal(getattr(oa, k), getattr(ob, k)), (step, k)
        va, vb = a.visits(), b.visits()
        assert np.array_equal(va[0], vb[0]) and np.array_equal(va[1], vb[1]), step
        if n <= 4000 and len(sizes) == 1:
            assert np.array_equal(va[0], [len(q) for q in lists]), step
    a.close()
    b.close()


@pytest.mark.parametrize("lanes", [16, 32, 64])
@pytest.mark.parametrize("n,patch", [(40, 0.04), (300, 0.1), (300, 0.01)])
def test_piled_particles(T, monkeypatch, lanes, n, patch):
    """Buckets of three to eight particles, read four states at a time, and fuller ones (a patch of a few
    vertices), in the shapes that walk lane by lane: raw and sorted buckets give the same bits and each
    particle's visited set has the size a plain kernel lists."""
    m, _ = P.mesh_and_tables(22, 0.1)
    rng = np.random.default_rng(n)
    x, y, th = ((0.5 + patch * (rng.random(n) - 0.5)).astype(np.float32) for _ in range(3))
    one = T.Sim(m, T.params(**P.PHYS, sigma=0.1), n)
    one.set_state(x, y, th)
    assert max(np.bincount(one.get_state().vid)) > 2
    sizes = [len(q) for q in one.neighbor_lists()]
    one.close()
    got = []
    for raw in (True, False):
        b = _batch(T, m, [n], raw, monkeypatch, lanes, x, y, th)
        b.stage_noise(np.zeros((1, n), np.float32))
        assert b.run(1, 0) == T.OK
        assert np.array_equal(b.visits()[0], sizes)
        got.append((b.get_state(), b.visits()[1]))
        b.close()
    for k in ("x", "y", "theta", "vid"):
        assert np.array_equal(getattr(got[0][0], k), getattr(got[1][0], k)), k
    assert np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("lanes", [1, 2, 4, 8])
@pytest.mark.parametrize("raw", [True, False])
@pytest.mark.parametrize("n,patch", [(1, 1.0), (65, 0.05), (300, 0.02), (1500, 1.0)])
def test_headings_by_the_whole_wave(T, monkeypatch, lanes, raw, n, patch):
    """Alignment sums redone in FP64 by the whole wave: random headings with dt / tau = 1, where a sum
    below 0.6 of its neighbours is redone, for one particle, for a few crowded buckets (300 particles
    on the vertices of a small patch: more than 8, and more than 64, in one) and for rows over several
    rounds of entries; raw and sorted buckets. Nothing moves (v0 = mu = 0), so each heading is the mean
    of its neighbours' in FP64: up to the FP32 rounding of the result where the sum is redone (2.4e-7 at
    2 pi), up to 1e-6 where it is left in FP32 (three roundings of that size and the sum's 1e-7)."""
    m, _ = P.mesh_and_tables(22, 0.1)
    phys = dict(P.PHYS, v0=0.0, mu=0.0, tau=P.PHYS["dt"])
    rng = np.random.default_rng(n)
    x, y = (0.5 + patch * (rng.random(n) - 0.5) for _ in range(2))
    th = rng.random(n) * 2 * np.pi
    x, y, th = (q.astype(np.float32) for q in (x, y, th))
    monkeypatch.setenv("TISSUE_SORTED_BUCKETS", "0" if raw else "1")
    b = T.Batch(m, [n], [T.params(**phys, sigma=0.1)])
    monkeypatch.delenv("TISSUE_SORTED_BUCKETS")
    b.set_mode(T.MODE_STEP_KERNEL)
    b.set_launch(lanes, 128)
    b.set_state(x, y, th)
    one = T.Sim(m, T.params(**phys, sigma=0.1), n)
    one.set_state(x, y, th)
    th64 = th.astype(np.float64)
    want = np.empty(n)
    tol = np.full(n, 1e-6)
    for i, js in enumerate(one.neighbor_lists()):
        c, s = np.cos(th64[js]).sum(), np.sin(th64[js]).sum()
        if np.hypot(c, s) < 0.59 * len(js):
            tol[i] = 2.5e-7
        want[i] = th64[i] + (np.arctan2(s, c) - th64[i] + np.pi) % (2 * np.pi) - np.pi
    assert (tol < 1e-6).sum() > n // 2 or n == 1
    b.stage_noise(np.zeros((1, n), np.float32))
    assert b.run(1, 0) == T.OK
    diff = (b.get_state().theta.astype(np.float64) - want + np.pi) % (2 * np.pi) - np.pi
    assert (np.abs(diff) <= tol).all(), np.abs(diff).max()
    one.close()
    b.close()


@pytest.mark.parametrize("lanes", [2, 8])
def test_full_workgroup_of_the_persistent_kernel(T, lanes):
    """Block 512 runs as 1,024 threads where the reduction words fit beside the replica, as 512 up to the
    capacity: states and outputs are the step kernel's at the same layout of the sums, bit for bit."""
    m, _ = P.mesh_and_tables(32, 0.05)
    cap = T.resident_capacity(m)
    prm = T.params(**P.PHYS, sigma=0.05)
    for n in (1, 64, 1025, cap - 24, cap):
        noise = T.gen_noise(3, 0.1, 2, n)
        got = []
        for mode, block in ((T.MODE_RESIDENT, 512), (T.MODE_RESIDENT, 256), (T.MODE_STEP_KERNEL, 256)):
            s = T.Sim(m, prm, n)
            s.set_mode(mode)
            s.set_launch(lanes, block)
            s.init_random(9)
            assert s.step(2, noise) == T.OK
            st, o = s.get_state(), s.get_outputs()
            got.append([st.x, st.y, st.theta, st.vid, o.vx, o.vy, o.r3d, o.face, o.nbr])
            phi = s.order()
            got[-1].append(phi[0])
            assert np.allclose(phi[1], got[0][10] if len(got) > 1 else phi[1], rtol=0, atol=1e-12)
            got[-1].append(phi[1])
            s.close()
        for other in got[1:]:
            for a, b in zip(got[0][:10], other[:10]):
                assert np.array_equal(a, b), n


@pytest.mark.parametrize("block", [64, 128, 512])
@pytest.mark.parametrize("n", [1, 100, 300])
def test_persistent_kernel_between_its_barriers(T, block, n):
    """Vertex counts scanned in registers (4,907 vertices: 5 a thread at 1,024 threads) and in LDS (39 and 77
    a thread), one pass over the replica and several (the last one's states held in registers), one wave and
    sixteen: states, neighbour counts and order parameters are the step kernel's, states and order parameters
    also where a step fails (the persistent kernel then writes no outputs of that run)."""
    m, _ = P.mesh_and_tables(22, 0.1)
    prm = T.params(**P.PHYS, sigma=0.1)
    for bad in (None, 2):
        noise = T.gen_noise(5, 0.1, 4, n)
        if bad is not None:
            noise[bad, n - 1] = np.nan
        got = []
        for mode, b in ((T.MODE_RESIDENT, block), (T.MODE_STEP_KERNEL, 128)):
            s = T.Sim(m, prm, n)
            s.set_mode(mode)
            s.set_launch(8, b)
            s.init_random(11)
            code = s.step(4, noise)
            st, o, phi = s.get_state(), s.get_outputs(), s.order()
            got.append((code, [st.x, st.y, st.theta, st.vid] + ([o.nbr] if bad is None else []), phi))
            s.close()
        (ca, a, pa), (cb, c, pb) = got
        assert ca == cb and (ca == T.OK) == (bad is None)
        for u, v in zip(a, c):
            assert np.array_equal(u, v, equal_nan=u.dtype.kind == "f"), (bad, n)
        k = 4 if bad is None else bad
        assert np.array_equal(pa[0][:k], pb[0][:k])
        assert np.allclose(pa[1][:k], pb[1][:k], rtol=0, atol=1e-12)
