"""The cell sort's temporaries: what the host asks for against the room that
the sort lays out, and against what the step without allocation had for it
when digits were 8 bits (4 ints a particle and 256 bins for each 4096)."""
import ctypes
import os

import pytest

from mpm_amd import capi


@pytest.fixture(scope="module")
def temp_ints():
    if not os.path.exists(capi.LIB_PATH):
        pytest.skip("libmpmx.so not built")
    f = ctypes.CDLL(capi.LIB_PATH)["_ZN4mpmx20radix_sort_temp_intsEli"]
    f.restype = ctypes.c_int64
    f.argtypes = [ctypes.c_int64, ctypes.c_int]
    return f


def _before(n):
    tiles = max((n + 4095) // 4096, 1)
    return 4 * n + 256 * tiles + (256 * tiles + 1023) // 1024 + 64


NS = [1, 255, 256, 257, 4095, 20000, 60000, 65535, 65536, 400000, 524287, 524288, 2097152, 10**7]


@pytest.mark.parametrize("n", NS)
def test_scratch_of_large_meshes_is_no_larger_than_it_was(temp_ints, n):
    """Ordered mode's cell ranges, 8 bytes a cell, are what makes a deck of few
    particles reach the 64 MiB: from 2^20 cells on (below, 65535 particles at
    the 704 bytes of ordered mode's largest set of options leave room) the sort
    asks for no more than before, up to the 2^23 cells that fill them."""
    assert 65535 * 704 + (1 << 20) * 8 < 64 << 20
    for cells in (1 << 20, (1 << 21) - 1, 1 << 21, 3000000, 8000000, 1 << 23):
        assert temp_ints(n, cells) <= _before(n), (n, cells)


@pytest.mark.parametrize("n", NS)
def test_scratch_holds_keys_ids_table_and_totals(temp_ints, n):
    for cells in (1, 2, 1023, 1024, 40000, 1048575, 1048576, 2**27):
        bits = max(cells.bit_length(), 1)  # keys 0 .. cells
        width = -(-bits // -(-bits // 10))
        per = 256 * (1 if n < 64 << 10 else 4 if n < 512 << 10 else 8 if n < 2 << 20 else 16)
        table = 2**width * -(-n // per)
        assert temp_ints(n, cells) >= 2 * n + table + -(-table // 1024), (n, cells)
