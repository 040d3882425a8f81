"""The block -> tile orders on lattices whose planes are no multiple of 8 tiles (site.h tile_site, host build): plane bands of
the nearest multiple and z slabs of uneven length visit every 64-site tile once."""
import ctypes

import numpy as np
import pytest

from tests.helpers import hostcheck_lib


@pytest.mark.parametrize("N", [(81, 75, 125), (90, 77, 20), (225, 250, 3), (48, 48, 7), (22, 66, 9), (36, 20, 64), (5, 3, 2)])
def test_ragged_orders_visit_every_tile_once(N):
    hc = hostcheck_lib()
    hc.hc_tile_sites.argtypes = [ctypes.POINTER(ctypes.c_int)] + [ctypes.c_int] * 6 + [ctypes.c_long,
                                                                                      ctypes.POINTER(ctypes.c_long)]
    P, S = N[0] * N[1], N[0] * N[1] * N[2]
    nt = (S + 63) // 64
    orders = [(3, nt // 8, 0, 0, nt % 8, 0)]
    if (P + 256) // 512:
        orders.append((1, (P + 256) // 512, 0, 0, 0, 0))
    for mode, bpb, bw, bh, nbx, tpbp in orders:
        out = np.zeros(nt, dtype=np.int64)
        hc.hc_tile_sites((ctypes.c_int * 3)(*N), mode, bpb, bw, bh, nbx, tpbp, nt, out.ctypes.data_as(ctypes.POINTER(ctypes.c_long)))
        assert np.array_equal(np.sort(out), np.arange(nt) * 64), (N, mode)
