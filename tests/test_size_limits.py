"""What is too large is refused when a simulation is created, before any device call: particles beyond the
32-bit byte offsets of the kernels, and meshes whose vertex ids do not fit the whole-wave walk's list; and, when
the tables are built, a geodesic table of more entries than 32-bit row numbers can name."""
import ctypes as C

import pytest

from test_device_math import H  # noqa: F401  (the host build, as a fixture)

P_MAX, V_MAX = (2**31 - 1) // 16, 2**26 - 1


@pytest.mark.parametrize("particles,vertices,refused", [(1, 1, 0), (P_MAX, V_MAX, 0), (P_MAX + 1, 1, 1), (1, V_MAX + 1, 1),
                                                        (2**40, 2**40, 1)])
def test_limits(H, particles, vertices, refused):  # noqa: F811
    H.hc_size_refused.argtypes = [C.c_long, C.c_long]
    assert H.hc_size_refused(particles, vertices) == refused


def test_creation_refuses_them(T):
    m = T.Mesh.ellipsoid(2.0, 1.0, 1.0, 4).build_tables(0.2)
    with pytest.raises(T.TissueError, match="too many particles") as e:
        T.Sim(m, T.params(sigma=0.1), P_MAX + 1)
    assert e.value.code == T.E_INVALID_ARG


@pytest.mark.parametrize("entries,refused", [(0, 0), (2**29, 0), (2**31 - 1 - 2**16, 0), (2**31 - 2**16, 1), (2**32 + 5, 1)])
def test_table_entries(H, entries, refused):  # noqa: F811
    H.hc_table_refused.argtypes = [C.c_int64]
    assert H.hc_table_refused(entries) == refused
