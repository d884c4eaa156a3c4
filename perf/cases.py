"""The work a program has this framework do, as cases that can be timed and compared.

Each case goes through the public entry points of ``2dtissue_amd``:

  update   one call of the drop-in class's update(): one step with a host noise row, then the state
           and the outputs read back (a program that plots or streams every step)
  run      a simulation from its initial state to its results: set_state, n steps, read-back of
           state, outputs and order history
  batch    an ensemble of replicas with sizes and parameters of their own, from initial states to
           results, at the launch shape the library picks (mode 0) or in the persistent kernel
           (mode 2, what parameter sweeps of equal replicas use)
  adjoint  gradients of a trajectory loss (forward, checkpoints, reverse) of one system or of an
           ensemble, the inner call of a parameter fit
  noalloc  one step on arrays that live on the GPU already (a serving loop that may not allocate)

The step is deterministic, so the same inputs give the same bits; it is also chaotic (a rounding
grows about 200-fold per step for particles that share a vertex), so only single steps have an
independent FP64 value to be compared with: ``exact`` gives it for update and noalloc.
"""
from __future__ import annotations

import ctypes as C
import functools
import importlib
import math

import numpy as np
import torch

T = importlib.import_module("2dtissue_amd")

# surfaces: ellipsoid with semi-axes (2, 1, 1), or a sphere of radius 1 + 0.2 Y_3^2
SURFACES = {
    "ellipsoid22": (22, 0.1),    # 4,907 UV vertices; the README's 100-particle example
    "ellipsoid32": (32, 0.05),   # 10,337 UV vertices; the 2,000-particle system
    "ellipsoid70": (70, 0.025),  # 49,211 UV vertices
    "sphere100": (100, 0.01),    # 100,265 UV vertices, 200,000 faces; 100,000 particles
}


@functools.lru_cache(maxsize=len(SURFACES))
def surface(name: str):
    freq, sigma = SURFACES[name]
    m = T.Mesh.perturbed_sphere(0.2, freq) if name.startswith("sphere") else T.Mesh.ellipsoid(2.0, 1.0, 1.0, freq)
    return m.build_tables(sigma)


def listed() -> list:
    return [
        # the smallest call: the README's example (100 particles), one update() at a time
        dict(name="update-100", kind="update", surface="ellipsoid22", n=100),
        # the same call on the 2,000-particle surface, an odd size
        dict(name="update-1999", kind="update", surface="ellipsoid32", n=1999),
        # one step on device arrays, no allocation (a serving loop)
        dict(name="noalloc-2000", kind="noalloc", surface="ellipsoid32", n=2000),
        # the README's whole run: 100 particles, 50 steps, noise from the host
        dict(name="run-100", kind="run", surface="ellipsoid22", n=100, steps=50),
        # the benchmark's system: 2,000 particles, 1,000 steps
        dict(name="run-2000", kind="run", surface="ellipsoid32", n=2000, steps=1000),
        # a middle size on a finer surface (sorted buckets), ragged against every tile size
        dict(name="run-9001", kind="run", surface="ellipsoid70", n=9001, steps=100),
        # the large surface: 100,000 particles
        dict(name="run-100000", kind="run", surface="sphere100", n=100000, steps=100),
        # the ensemble of the benchmark: 256 replicas of 100 to 4,000 particles
        dict(name="batch-256", kind="batch", surface="ellipsoid32", replicas=256, lo=100, hi=4000, steps=200, mode=0),
        # a small ragged ensemble at the library's own choice of mode
        dict(name="batch-37", kind="batch", surface="ellipsoid32", replicas=37, lo=17, hi=699, steps=100, mode=0),
        # a parameter sweep: 256 equal replicas of 200 in the persistent kernel
        dict(name="sweep-256", kind="batch", surface="ellipsoid32", replicas=256, lo=200, hi=200, steps=100, mode=2),
        # gradients of the 1,000-particle system over 200 steps
        dict(name="adjoint-1000", kind="adjoint", surface="ellipsoid32", replicas=1, lo=1000, hi=1000, steps=200),
        # gradients of 64 x 2,000 particles on the large surface
        dict(name="adjoint-64x2000", kind="adjoint", surface="sphere100", replicas=64, lo=2000, hi=2000, steps=200),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _surface_for(n: int) -> str:
    return "ellipsoid22" if n <= 400 else "ellipsoid32" if n <= 4000 else "ellipsoid70" if n <= 20000 else "sphere100"


def draw(rng) -> dict:
    kind = rng.choice(("update", "noalloc", "run", "run", "run", "batch", "batch", "sweep", "adjoint", "adjoint"))
    if kind in ("update", "noalloc"):
        n = _log_int(rng, 60, 100000 if kind == "update" else 4000)
        return dict(kind=kind, surface=_surface_for(n), n=n)
    if kind == "run":
        n = _log_int(rng, 50, 100000)
        return dict(kind=kind, surface=_surface_for(n), n=n, steps=_log_int(rng, 10, 400 if n <= 20000 else 100))
    if kind == "batch":
        hi = _log_int(rng, 150, 4000)
        return dict(kind="batch", surface="ellipsoid32", replicas=_log_int(rng, 2, 256), lo=max(1, hi // rng.randint(2, 40)),
                    hi=hi, steps=_log_int(rng, 10, 150), mode=0)
    if kind == "sweep":
        n = _log_int(rng, 40, 600)
        return dict(kind="batch", surface="ellipsoid32", replicas=rng.randint(100, 256), lo=n, hi=n,
                    steps=_log_int(rng, 10, 100), mode=2)
    if rng.random() < 0.5:
        n = _log_int(rng, 100, 4000)
        return dict(kind="adjoint", surface=_surface_for(n), replicas=1, lo=n, hi=n, steps=_log_int(rng, 10, 200))
    hi = _log_int(rng, 100, 2000)
    return dict(kind="adjoint", surface=rng.choice(("ellipsoid32", "sphere100")), replicas=rng.randint(2, 60),
                lo=max(1, hi // rng.randint(1, 8)), hi=hi, steps=_log_int(rng, 10, 150))


def _sizes(case: dict) -> np.ndarray:
    """The replicas' sizes: uniform in [lo, hi], the same for every seed."""
    return np.random.default_rng(3).integers(case["lo"], case["hi"] + 1, case["replicas"])


def _params(case: dict, tau: float = 1.0, v0: float = 1.0):
    return T.params(sigma=SURFACES[case["surface"]][1], v0=v0, k=10.0, mu=1.0, tau=tau, dt=0.02)


def _noise(rng, rows: int, n: int) -> np.ndarray:
    return (0.1 * rng.standard_normal((rows, n), dtype=np.float32)).astype(np.float32)


def prepare(case: dict, seed: int) -> dict:
    mesh = surface(case["surface"])
    rng = np.random.default_rng([seed, 77])
    kind = case["kind"]
    if kind in ("update", "run", "noalloc"):
        n, p = case["n"], _params(case)
        x, y, th = mesh.random_init_host(seed, n)
        sim = T.Sim(mesh, p, n)
        s = dict(kind=kind, sim=sim, n=n, x=x, y=y, th=th)
        if kind == "update":
            sim.set_state(x, y, th)
            s.update(noise=_noise(rng, 64, n), t=0)
        elif kind == "run":
            s.update(steps=case["steps"], noise=_noise(rng, case["steps"], n), host_noise=n <= 400)
            if not s["host_noise"]:
                sim.stage_noise(s["noise"])
        else:
            sim.set_state(x, y, th)
            dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
            f = lambda: torch.empty(n, dtype=torch.float32, device="cuda")  # noqa: E731
            i = lambda: torch.empty(n, dtype=torch.int32, device="cuda")  # noqa: E731
            s.update(p=p, mesh=mesh, ins=[dev(x), dev(y), dev(th), dev(sim.get_state().vid)], eta=dev(_noise(rng, 64, n)[0].copy()),
                     outs=dict(x=f(), y=f(), theta=f(), vid=i(), vx=f(), vy=f(), r3x=f(), r3y=f(), r3z=f(), face=i(),
                               nbr=i(), phi=torch.empty(2, dtype=torch.float64, device="cuda"),
                               flags=torch.empty(1, dtype=torch.int32, device="cuda")))
        return s
    sizes = _sizes(case)
    R = len(sizes)
    if kind == "adjoint":
        ps = [_params(case)] * R
    else:
        g = np.random.default_rng(4)
        tau, v0 = np.exp(g.uniform(np.log(0.1), np.log(10.0), R)), g.uniform(0.5, 2.0, R)
        ps = [_params(case, float(tau[r]), float(v0[r])) for r in range(R)]
    start = [mesh.random_init_host(1000 * seed + r, int(sizes[r])) for r in range(R)]
    x, y, th = (np.concatenate([q[k] for q in start]) for k in range(3))
    single = kind == "adjoint" and R == 1
    h = T.Sim(mesh, ps[0], int(sizes[0])) if single else T.Batch(mesh, sizes, ps)
    s = dict(kind=kind, h=h, x=x, y=y, th=th, steps=case["steps"], replicas=R)
    if kind == "batch":
        if case["mode"]:
            h.set_mode(case["mode"])
        std = np.random.default_rng(5).uniform(0.0, 0.5, R)
        h.gen_noise(np.arange(R, dtype=np.uint64) + 1000 * seed, std, case["steps"])
    else:
        h.stage_noise(_noise(rng, case["steps"], len(x)))
        s["loss"] = T.loss(target_order=0.8, w_order=1.0, w_velocity=0.1, modes=T.target_field())
    return s


def _ok(code: int) -> None:
    if code != T.OK:
        raise RuntimeError(f"status {code}")


def _results(h) -> dict:
    st, o = h.get_state(), h.get_outputs()
    return dict(x=st.x, y=st.y, theta=st.theta, vid=st.vid, vx=o.vx, vy=o.vy, r3d=o.r3d, face=o.face, nbr=o.nbr)


def run(s: dict):
    kind = s["kind"]
    if kind == "update":
        row = s["noise"][s["t"] % len(s["noise"])]
        s["t"] += 1
        _ok(s["sim"].step(1, row))
        return _results(s["sim"])
    if kind == "run":
        sim = s["sim"]
        sim.reset_order()
        sim.set_state(s["x"], s["y"], s["th"])
        _ok(sim.step(s["steps"], s["noise"]) if s["host_noise"] else sim.step_staged(s["steps"], 0))
        out = _results(sim)
        out["phi_ref"], out["phi_polar"] = sim.order()
        return out
    if kind == "noalloc":
        o = s["outs"]
        order = ("x", "y", "theta", "vid", "vx", "vy", "r3x", "r3y", "r3z", "face", "nbr", "phi", "flags")
        ptr = [C.c_void_p(t.data_ptr()) for t in (*s["ins"], s["eta"], *(o[k] for k in order))]
        _ok(T.lib().tissue_step_noalloc(s["mesh"].h, C.byref(s["p"]), s["n"], *ptr,
                                        C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        return o
    h = s["h"]
    h.set_state(s["x"], s["y"], s["th"])
    if kind == "batch":
        _ok(h.run(s["steps"], 0))
        return _results(h)
    code, g, dth, dx, dy = h.adjoint(s["steps"], s["loss"], first_row=0, ckpt_every=20)
    _ok(code)
    g = g if isinstance(g, list) else [g]
    out = {k: np.array([q[k] for q in g]) for k in g[0] if not k.endswith("_ms")}
    out.update(d_theta0=dth, d_x0=dx, d_y0=dy, state=_results(h))
    return out


def work(case: dict) -> dict:
    """64 bytes per particle-step (x, y, theta, vertex id and noise read; x, y, theta, vx, vy, r3d,
    vertex id, face and neighbour count written), twice that with its reverse; about 270 operations
    (20 per neighbour pair, 40 per particle, 40 per candidate face of the remap)."""
    n = int(_sizes(case).sum()) if "replicas" in case else case["n"]
    ps = n * case.get("steps", 1)
    both = 2 if case["kind"] == "adjoint" else 1
    return dict(bytes=64 * ps * both, flops=270 * ps * both)


# ------------------------------------------------------------------ one step in 64 bits

def _cross2(ax, ay, bx, by):
    return ax * by - ay * bx


def _locate(e: dict, px, py):
    """The face nearest to each point (the lowest id where several are), the 3-D point blended from its
    corners with the distances to them as weights, and the corner nearest to that point."""
    tri = e["uv"][e["faces"]]                       # [F, 3, 2]
    lo, hi = tri.min(1) - 1e-12, tri.max(1) + 1e-12
    face = np.zeros(len(px), np.int64)
    for c in range(0, len(px), 256):
        x, y = px[c:c + 256, None], py[c:c + 256, None]
        i, f = np.nonzero((x >= lo[:, 0]) & (x <= hi[:, 0]) & (y >= lo[:, 1]) & (y <= hi[:, 1]))
        p = np.stack([px[c + i], py[c + i]], 1)
        a, b, q = tri[f, 0], tri[f, 1], tri[f, 2]
        area = _cross2(*(b - a).T, *(q - a).T)
        inside = np.minimum(np.minimum(_cross2(*(b - a).T, *(p - a).T) / area, _cross2(*(q - b).T, *(p - b).T) / area),
                            _cross2(*(a - q).T, *(p - q).T) / area)
        inside = np.minimum(inside, 0.0)            # how far outside, 0 inside
        order = np.lexsort((f, -inside, i))
        i, f = i[order], f[order]
        first = np.r_[True, i[1:] != i[:-1]]
        face[c + i[first]] = f[first]
    corner = e["faces"][face]
    w = np.hypot(px[:, None] - e["uv"][corner, 0], py[:, None] - e["uv"][corner, 1])
    w /= w.sum(1, keepdims=True)
    X = e["xyz"].astype(np.float32).astype(np.float64)[corner]
    r3 = (w[:, :, None] * X).sum(1)
    near = np.argmin(np.linalg.norm(r3[:, None, :] - X, axis=2), axis=1)
    return face, corner[np.arange(len(px)), near], r3


def _seam_wrap(ax, ay, px, py):
    """The reference's restart loop per particle: the first of left, right, up, down that the move
    crosses, its gluing map on the end point, the swapped exit point as the next start."""
    ax, ay, px, py = (np.array(v, np.float64) for v in (ax, ay, px, py))
    turn = np.zeros(len(px))
    for _ in range(16384):
        k = np.nonzero(~((px >= 0) & (px <= 1) & (py >= 0) & (py <= 1)))[0]
        if not len(k):
            return px, py, turn
        a, b, x, y = ax[k], ay[k], px[k], py[k]
        dx, dy = x - a, y - b
        side = np.full(len(k), 4)
        t = np.zeros(len(k))
        with np.errstate(divide="ignore", invalid="ignore"):
            for q, (cx, cy, ex, ey) in enumerate(((0, 0, 0, 1), (1, 0, 0, 1), (0, 1, 1, 0), (0, 0, 1, 0))):
                det = dx * ey - dy * ex
                tq = ((cx - a) * ey - (cy - b) * ex) / det
                sq = ((cx - a) * dy - (cy - b) * dx) / det
                on = ((a == cx) & (b >= 0) & (b <= 1)) if ex == 0 else ((b == cy) & (a >= 0) & (a <= 1))
                hit = (side == 4) & ~on & (np.abs(det) >= 1e-9) & (tq >= 0) & (tq <= 1) & (sq >= 0) & (sq <= 1)
                side[hit], t[hit] = q, tq[hit]
        ex, ey = a + t * dx, b + t * dy
        ex = np.where(np.abs(ex) < 1e-3, 0.0, ex)
        ey = np.where(np.abs(ey) < 1e-3, 0.0, ey)
        ex, ey = np.where(side == 4, a, ex), np.where(side == 4, b, ey)
        px[k] = np.choose(side, (y, y, 2 - y, -y, -y))
        py[k] = np.choose(side, (-x, 2 - x, x, x, x))
        turn[k] -= np.where(side <= 1, 0.5, 1.5) * np.pi
        ax[k], ay[k] = ey, ex
    return px, py, turn


def exact(case: dict, seed: int):
    if case["kind"] not in ("update", "noalloc") or case["n"] > 20000:
        return None
    mesh = surface(case["surface"])
    e = mesh.export()
    n, sigma = case["n"], SURFACES[case["surface"]][1]
    x, y, th = (v.astype(np.float64) for v in mesh.random_init_host(seed, n))
    eta = _noise(np.random.default_rng([seed, 77]), 64, n)[0].astype(np.float64)
    _, vid, _ = _locate(e, x, y)
    # pairs (i, j) and their table distances: the particles on the vertices of row vid[i]
    by_vertex = np.argsort(vid, kind="stable")
    count = np.bincount(vid, minlength=e["nv"])
    start = np.r_[0, np.cumsum(count)[:-1]]
    rows = e["row_ptr"][vid + 1] - e["row_ptr"][vid]
    i = np.repeat(np.arange(n), rows)
    ent = np.repeat(e["row_ptr"][vid], rows) + np.arange(len(i)) - np.repeat(np.cumsum(rows) - rows, rows)
    m = count[e["col"][ent]]
    pi, pe = np.repeat(i, m), np.repeat(ent, m)
    pj = by_vertex[np.repeat(start[e["col"][ent]], m) + np.arange(len(pi)) - np.repeat(np.cumsum(m) - m, m)]
    d = e["dist"][pe].astype(np.float64)
    nbr = np.bincount(pi[(d != 0) & (d <= 2.4 * sigma)], minlength=n)
    near = d < 2 * sigma
    pi, pj, d = pi[near], pj[near], np.where(d[near] == 0, 0.001, d[near])
    c = np.where(pi != pj, -10.0 * (2 * sigma - d) / (2 * sigma) / d, 0.0)
    F = np.hypot(np.bincount(pi, c * (x[pi] - x[pj]), n), np.bincount(pi, c * (y[pi] - y[pj]), n))
    mean = np.arctan2(np.bincount(pi, np.sin(th[pj]), n), np.bincount(pi, np.cos(th[pj]), n))
    v = 1.0 + F
    vx, vy = v * np.cos(th), v * np.sin(th)
    delta = mean - th
    delta = np.where(delta > np.pi, delta - 2 * np.pi, np.where(delta <= -np.pi, delta + 2 * np.pi, delta))
    nx, ny, turn = _seam_wrap(x, y, x + 0.02 * vx, y + 0.02 * vy)
    nth = th + 0.02 * delta + eta + turn
    nth -= 2 * np.pi * np.floor((nth + np.pi) / (2 * np.pi))
    # the point is located where it is stored, in 32 bits
    face, nvid, r3 = _locate(e, nx.astype(np.float32).astype(np.float64), ny.astype(np.float32).astype(np.float64))
    out = dict(x=nx, y=ny, theta=nth, vid=nvid.astype(np.int32), vx=vx, vy=vy, face=face.astype(np.int32), nbr=nbr.astype(np.int32))
    if case["kind"] == "update":
        out["r3d"] = r3
        return out
    phi = [abs(np.sign(nx * vy - ny * vx).sum()) / n, math.hypot(np.cos(nth).sum(), np.sin(nth).sum()) / n]
    out.update(r3x=r3[:, 0], r3y=r3[:, 1], r3z=r3[:, 2], phi=np.array(phi), flags=None)
    return out
