"""The plan of the deviation kernel that walks z (site.h cg_walk_plan; host build): the blocks cover every unit of every chunk,
their partial sums have places, and with the x transforms every block is whole."""
import ctypes
import itertools

from tests.helpers import hostcheck_lib


def plan(N, xf, forced):
    out = (ctypes.c_long * 2)()
    hostcheck_lib().hc_cg_walk((ctypes.c_int * 3)(*N), ctypes.c_int(xf), ctypes.c_int(forced), out)
    return out[0], out[1]


def test_plan_covers_the_lattice():
    taken = 0
    for N in itertools.product((1, 16, 25, 31, 64, 100, 125, 128), (1, 8, 33, 40, 75, 100, 128), (1, 2, 5, 64, 100, 250, 384)):
        P, units = N[0] * N[1], (N[0] * N[1] + 255) // 256
        for xf, forced in itertools.product((0, 1), (-1, 0, 1, 4, 7, 32)):
            zc, n = plan(N, xf, forced)
            if zc == 0:
                assert n == 0
                continue
            taken += 1
            assert forced and (forced < 0 or zc == forced)
            assert n == units * ((N[2] + zc - 1) // zc) <= (P * N[2] + 255) // 256
            assert not xf or P % 256 == 0
    assert taken > 500


def test_ragged_planes_of_several_units_walk():
    """The form that 100 x 100 x 100 and 125 x 125 x 250 take by themselves."""
    for N in ((100, 100, 100), (125, 125, 250)):
        zc, n = plan(N, 0, -1)
        assert zc > 0 and N[0] * N[1] % 256 and n % ((N[0] * N[1] + 255) // 256) == 0
