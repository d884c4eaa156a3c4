"""The closed form of the seam wrap (seam_fold in 2dtissue_amd/csrc/geom.h) against the loop it stands
for (EuclideanTiling::diagonal_seam_edges_square_border, EuclideanTiling.cpp:31-69), on the host build
of the device geometry: wherever it settles a move, the FP32 position and heading and the quarter turns
are the loop's, exactly; wherever it does not, it leaves its arguments alone."""
import ctypes as C

import numpy as np
import pytest

from test_device_math import H, p  # noqa: F401  (the host build, as a fixture)


def flights(seed, n, lo, hi, single):
    """Starts anywhere, on edges, in corners and within the exit snapping's 1e-3 of them; moves of
    length lo..hi in any direction, some along the axes and diagonals."""
    rng = np.random.default_rng(seed)
    a = rng.random((n, 2)).astype(np.float32).astype(np.float64)
    k = np.arange(n) % 9
    a[k == 1, 0] = 0.0
    a[k == 2, 1] = 1.0
    a[k == 3] = 0.0
    a[k == 4] = 1.0
    a[k == 5] = (0.0, 1.0)
    a[k == 6] *= 2e-3
    a[k == 7] = 1.0 - 2e-3 * a[k == 7]
    a = a.astype(np.float32).astype(np.float64)
    length = np.exp(rng.uniform(np.log(lo), np.log(hi), n))
    ang = rng.uniform(-np.pi, np.pi, n)
    special = rng.random(n) < 0.1
    ang[special] = np.round(ang[special] * 4 / np.pi) * np.pi / 4 + rng.choice([0.0, 1e-3, -1e-4], special.sum())
    b = a + length[:, None] * np.stack([np.cos(ang), np.sin(ang)], 1)
    if single:  # a small step's end point is a sum of FP32 values
        b = b.astype(np.float32).astype(np.float64)
    th = rng.uniform(-np.pi, np.pi, n)
    th[::2] = th[::2].astype(np.float32)
    out = ~((b >= 0) & (b <= 1)).all(1)
    return a[out].copy(), b[out].copy(), th[out].copy()


def both(H, a, b, th, maxc):  # noqa: F811
    n = len(a)
    r = b.copy(); dth = np.zeros(n); ok = np.zeros(n, np.int32); cr = np.zeros(n, np.int32); q = np.zeros(n, np.int32)
    H.hc_seam_wrap_many(n, p(a, C.c_double), p(b, C.c_double), maxc, p(r, C.c_double), p(dth, C.c_double),
                        p(ok, C.c_int32), p(cr, C.c_int32))
    H.hc_seam_wrap_quarter_many(n, p(a, C.c_double), p(b, C.c_double), maxc, p(q, C.c_int32))
    H.hc_wrap_heading.argtypes, H.hc_wrap_heading.restype = [C.c_double], C.c_double
    t = np.array([H.hc_wrap_heading(v) for v in th + dth])
    fb, ft = b.copy(), th.copy()
    st = np.zeros(n, np.int32); fq = np.full(n, -1, np.int32)
    H.hc_seam_fold_many(n, p(a, C.c_double), p(fb, C.c_double), p(ft, C.c_double), maxc, p(st, C.c_int32), p(fq, C.c_int32))
    return r, t, ok, cr, q, fb, ft, st.astype(bool), fq


@pytest.mark.parametrize("lo,hi,single,least", [(1e-4, 1.5, True, 0.9), (1e-2, 40.0, False, 0.9), (40.0, 600.0, False, 0.8)])
def test_fold_is_the_loop_in_fp32(H, lo, hi, single, least):  # noqa: F811
    a, b, th = flights(21, 60000, lo, hi, single)
    r, t, ok, cr, q, fb, ft, st, fq = both(H, a, b, th, 16384)
    assert ok.all()
    f32 = np.float32
    assert np.array_equal(fb[st].astype(f32), r[st].astype(f32))
    assert np.array_equal(ft[st].astype(f32), t[st].astype(f32))
    assert np.array_equal(fq[st], q[st])
    assert np.array_equal(fb[~st], b[~st]) and np.array_equal(ft[~st], th[~st]) and (fq[~st] == -1).all()
    assert st.mean() > least  # it is the path that runs, not the exception


def test_fold_leaves_doubtful_moves_to_the_loop(H):  # noqa: F811
    # end points whose image lies on the border, within 1e-9 of it, or in a corner
    e = np.array([0.0, 1e-10, -1e-10])
    for x in (-3.0, 2.0, 5.0):
        for dx in e:
            b = np.array([[x + dx, 0.3], [0.3, x + dx], [x + dx, x + dx]])
            *_, st, _ = both(H, np.full((3, 2), 0.5), b, np.full(3, 0.1), 16384)
            assert not st.any(), (x, dx)
    # a heading that lands on +-pi, and one whose size leaves no FP32 certainty
    b = np.array([[1.25, 0.5], [1.25, 0.5], [1.25, 0.5]])
    th = np.array([np.pi / 2 - 1e-15, 0.3, 1e9])
    *_, st, _ = both(H, np.full((3, 2), 0.5), b, th, 16384)
    assert st.tolist() == [False, True, False]
    # non-finite values
    for bad in (np.inf, -np.inf, np.nan):
        st = np.zeros(1, np.int32); fq = np.zeros(1, np.int32)
        fb = np.array([[bad, 0.5]]); ft = np.array([0.1])
        H.hc_seam_fold_many(1, p(np.full((1, 2), 0.5), C.c_double), p(fb, C.c_double), p(ft, C.c_double), 16384,
                            p(st, C.c_int32), p(fq, C.c_int32))
        assert st[0] == 0


@pytest.mark.parametrize("maxc", [1, 63, 64, 67, 68, 100, 400])
def test_fold_respects_the_crossing_bound(H, maxc):  # noqa: F811
    """A move that the loop would report as not converging is never settled by the closed form."""
    a, b, th = flights(22, 20000, 1e-3, 120.0, False)
    r, t, ok, cr, q, fb, ft, st, fq = both(H, a, b, th, maxc)
    assert not st[ok == 0].any()
    length = np.abs(b - a).sum(1) + 16.0
    assert not st[4.0 * length > maxc].any()
    if maxc >= 100:
        assert st.any()
