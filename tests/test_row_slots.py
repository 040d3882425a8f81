"""The row copy of the step (site.h row_slots, halo_site; host build): for every lattice width and tile position the slots
of x + 1 and x - 1 hold the periodic neighbours in the site's own row, and every halo site lies on the lattice."""
import ctypes

import numpy as np
import pytest

from tests.helpers import hostcheck_lib


@pytest.mark.parametrize("nx", list(range(1, 132)) + [191, 192, 200, 255, 257, 511])
def test_row_copy_holds_the_periodic_neighbours(nx):
    f = hostcheck_lib().hc_row_neighbours
    lp = ctypes.POINTER(ctypes.c_long)
    f.argtypes = [ctypes.POINTER(ctypes.c_int), ctypes.c_long, lp, lp]
    for ny, nz in ((3, 2), (5, 1), (64, 1)):
        S = nx * ny * nz
        s = np.arange(S)
        row, x = s - s % nx, s % nx
        xp, xm = np.zeros(64, np.int64), np.zeros(64, np.int64)
        for first in range(0, S, 64):
            f((ctypes.c_int * 3)(nx, ny, nz), first, xp.ctypes.data_as(lp), xm.ctypes.data_as(lp))
            n = min(64, S - first)
            t = slice(first, first + n)
            assert np.array_equal(xp[:n], row[t] + (x[t] + 1) % nx), (nx, ny, first)
            assert np.array_equal(xm[:n], row[t] + (x[t] - 1) % nx), (nx, ny, first)
