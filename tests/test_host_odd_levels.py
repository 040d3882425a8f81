"""The initial state's own transforms take the variant compiled for the odd primes that their lengths have (fft_lds.h
odd_level), as every other transform does."""
import pytest

from tests import fake_runtime

SCRIPT = """
N = {N}
xl, xr = Glasma.draw_charges(1, N[0], N[1], 0.5, 0.5)
with Glasma(N) as g:
    g.mv_initial_state(0, Glasma.mv_params(1.65, 0.1, 2.0, 2.0, 2, 4), xl, xr)
for kernel in (b"k_sheet_plane", b"k_sheet_jinv"):
    print(*(fake.fake_launches_of(kernel + b"ILi%dE" % level) for level in range(3)))
"""


@pytest.mark.parametrize("N,plane,z", [((16, 12, 24), 0, 0), ((1, 1, 1), 0, 0), ((20, 12, 32), 1, 0), ((9, 14, 16), 1, 0),
                                       ((16, 16, 35), 0, 1), ((22, 16, 13), 2, 2), ((10, 13, 7), 2, 1), ((8, 8, 11), 0, 2)])
def test_variant_follows_the_lengths(N, plane, z):
    got = [[int(n) > 0 for n in line.split()] for line in fake_runtime.run(SCRIPT.format(N=N)).splitlines()]
    assert got == [[level == want for level in range(3)] for want in (plane, z)]
