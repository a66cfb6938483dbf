"""The tables of compiled demag kernels do not change after the library is
loaded.  Plan creation looks every candidate length up in them, registered or
not, while other threads may be reading: a look-up that added an entry would
rebalance the tree under them.  Without a GPU a plan fails on its first
allocation, which comes after the look-ups."""
import ctypes as C
import os

import pytest

from hotspin_amd import _lib

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="library not built")

# axis-1 columns of 2048 and of 4 points, rows of 3, 7 and 1280 points, run-time
# lengths: none of them in every table
MESHES = [(1, 1024, 1024), (1, 2, 8), (2, 8, 3), (3, 16, 7), (1, 16, 1100), (11, 13, 17), (200, 5, 3)]


def test_plans_of_unregistered_lengths_add_no_entry():
    L = _lib.lib()
    before = L.hs_demag_registered()
    assert before > 100  # five tables, about 30 lengths each
    cell, pbc = (C.c_double * 3)(2e-9, 2e-9, 2e-9), (C.c_int * 3)(0, 0, 0)
    for N in MESHES:
        d = L.hs_demag_create((C.c_int * 3)(*N), cell, pbc, 6, None)
        L.hs_clear_error()
        if d:
            L.hs_demag_destroy(d)
        assert L.hs_demag_registered() == before, N
