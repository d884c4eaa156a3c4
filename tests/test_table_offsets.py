"""The geodesic table's entries as the kernels address them (table_entry in 2dtissue_amd/csrc/geom.h), on the
host build: right on both sides of a 32-bit byte offset (2^29 entries of 8 bytes) and up to the last entry an
int can name. The table is a sparse mapping, of which only the pages around the tested entries exist."""
import ctypes as C
import mmap

import pytest

from test_device_math import H  # noqa: F401  (the host build, as a fixture)

MAP_NORESERVE = 0x4000


@pytest.mark.parametrize("entry", [0, 2**28, 2**29 - 1, 2**29, 2**29 + 5, 2**30, 2**31 - 1])
def test_entries_beyond_4_gib(H, entry):  # noqa: F811
    table = mmap.mmap(-1, 8 * 2**31, flags=mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS | MAP_NORESERVE)
    view = (C.c_int32 * 2).from_buffer(table, 8 * entry)
    view[0], view[1] = entry, ~entry
    base = (C.c_char * 1).from_buffer(table)
    out = (C.c_int32 * 2)()
    H.hc_table_entry(base, entry, out)
    got = (out[0], out[1])
    del view, base
    table.close()
    assert got == (entry, ~entry)
