"""Workgroups with waves past their replica's last particle, and waves partly past it: the block size decides how
many there are and changes no result. Replicas from one particle to a little over a tile, at every lane count
with whole-wave walks and at wider ones; one replica stopped by a failed step beside the others."""
import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu

SIZES = [1, 30, 31, 32, 33, 63, 64, 65, 127, 129, 2]


@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16, 64])
@pytest.mark.parametrize("copies", [1, 400])  # few particles (more physical lanes than the layout's), and many
def test_blocks_give_the_same_step(T, lanes, copies):
    m, _ = P.mesh_and_tables(32, 0.05)
    sizes = SIZES * copies
    R, n = len(sizes), sum(sizes)
    ps = [T.params(**P.PHYS, sigma=0.05)] * R
    ps[1] = T.params(**dict(P.PHYS, v0=1e30), sigma=0.05)  # leaves the crossing bound behind: stopped
    b = T.Batch(m, sizes, ps)
    b.set_mode(T.MODE_STEP_KERNEL)
    b.init_random(np.arange(R, dtype=np.uint64))
    s0 = b.get_state()
    b.stage_noise(np.random.default_rng(5).normal(0, 0.1, (3, n)).astype(np.float32))
    ref = None
    for block in (64, 128, 256, 512):
        b.set_launch(lanes, block)
        b.set_state(s0.x, s0.y, s0.theta, s0.vid)
        assert b.run(3, 0) != T.OK
        s, o, f = b.get_state(), b.get_outputs(), b.flags()[0]
        assert f[1] != 0 and not f[2:].any() and f[0] == 0
        got = [s.x, s.y, s.theta, s.vid] + [b.order(r)[k][-3:] for r in range(len(SIZES)) for k in (0, 1)]
        keep = np.ones(n, bool)
        keep[sizes[0]:sizes[0] + sizes[1]] = False  # a stopped replica writes no outputs
        got += [a[keep] for a in (o.vx, o.vy, o.r3d, o.face, o.nbr)]
        for a, c in zip(ref or got, got):
            assert np.array_equal(a, c), block
        ref = ref or got
    b.close()
