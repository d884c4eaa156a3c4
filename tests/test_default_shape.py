"""The default launch shape of the step kernel (tiled_default_shape, phys_lanes in 2dtissue_amd/csrc/launch.h): at
the edges of its rules, and over the whole range a shape the kernels are built for."""
import numpy as np
import pytest

from test_device_math import H, p  # noqa: F401  (the host build, as a fixture)
import ctypes as C

BUILT = {(1, 1), (2, 2), (2, 4), (4, 4), (4, 8), (8, 8), (8, 16), (16, 16), (32, 32), (64, 64)}


def shape(H, R, ntot, nmax, nv):  # noqa: F811
    out = np.zeros(4, np.int32)
    H.hc_default_shape(R, ntot, nmax, nv, p(out, C.c_int32))
    return tuple(int(v) for v in out)


@pytest.mark.parametrize("R,n,nv,want", [
    (1, 4096, 10337, (32, 64, 32)), (1, 4097, 10337, (8, 128, 16)), (1, 8193, 49211, (4, 128, 8)),
    (1, 100000, 100265, (4, 128, 4)), (2, 2048, 10337, (32, 64, 32)),
    # replicas that fill a workgroup of 128 or less; that fit in one of 256; that need more
    (1600, 64, 10337, (2, 128, 2)), (1600, 65, 10337, (2, 256, 2)), (800, 128, 10337, (2, 256, 2)),
    (800, 129, 10337, (2, 128, 2)), (1500, 33, 10337, (4, 256, 4)), (780, 64, 10337, (4, 256, 4)),
    (780, 65, 10337, (4, 128, 4)), (600, 17, 10337, (4, 256, 8)), (600, 33, 10337, (4, 128, 8)),
    # four lanes on four or eight, by particles and by the largest replica
    (384, 64, 10337, (4, 128, 8)), (385, 64, 10337, (4, 256, 4)), (500, 65, 10337, (4, 128, 8)),
])
def test_rules_edges(H, R, n, nv, want):  # noqa: F811
    assert shape(H, R, R * n, n, nv)[:3] == want


def test_every_shape_is_built_and_fits(H):  # noqa: F811
    rng = np.random.default_rng(1)
    for _ in range(20000):
        R = int(np.exp(rng.uniform(0, np.log(20000))))
        n = int(np.exp(rng.uniform(0, np.log(200000))))
        if R * n > 2**27 - 1:
            continue
        nv = int(np.exp(rng.uniform(np.log(10), np.log(1e6))))
        lanes, block, phys, lds = shape(H, R, R * n, n, nv)
        assert (lanes, phys) in BUILT and block in (64, 128, 256) and lds <= 65536, (R, n, nv)
