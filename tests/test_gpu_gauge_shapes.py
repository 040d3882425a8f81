"""Gauge fixing on lattices at the edges of the deviation kernel's and the transforms' rules: the z-walking deviation
kernel against the other one, and transforms against numpy.

Ragged planes (not a multiple of 256 sites: the last unit of a plane is partly empty), one and several chunks, a last
chunk that is short, both z boundaries; strided line groups of 4 up to 64 lines.  Tolerance between the two kernels 1e-12
(the same sums, grouped differently, a few hundred roundings of order-one terms).  The "fourier" update is left out: for
Nz > 1 it rotates every site by V mean(Delta), so each update multiplies the round-off by the number of sites and the
two kernels' results part as any two groupings of those sums do; the same kernel runs under "jacobi".
"""
import numpy as np
import pytest

from tests.helpers import random_fields, upload

pytestmark = pytest.mark.gpu
A = (1.0, 0.9, 0.8)


def _fixed(N, bc, f, algorithm, iters):
    from soerenpragya3dglasma_amd import Glasma
    with Glasma(N, A, 0.1, bc) as g:
        upload(g, f)
        stats = g.coulomb_gauge_algorithm(algorithm, 0.0, iters)
        UG, EG, G = g.get_gauge_fixed()
    return np.array(stats), np.asarray(UG), np.asarray(EG), np.asarray(G)


@pytest.mark.parametrize("N,bc", [((31, 8, 9), 0), ((15, 17, 5), 1), ((63, 4, 7), 0), ((32, 8, 6), 1), ((33, 39, 4), 0),
                                  ((1, 250, 6), 0)])
@pytest.mark.parametrize("algorithm", ["consistent", "jacobi"])
def test_walk_matches_other_kernel(monkeypatch, N, bc, algorithm):
    if algorithm == "consistent":  # transform lengths
        N = {31: (30, 9, 9), 15: (15, 18, 5), 63: (63, 4, 7), 32: (32, 8, 6), 33: (33, 39, 4), 1: (1, 250, 6)}[N[0]]
    f = random_fields(N, seed=sum(N), link_scale=0.2, bc=bc)
    monkeypatch.setenv("GLASMA_CG_WALK", "0")
    s0, U0, E0, G0 = _fixed(N, bc, f, algorithm, 4)
    for chunk in ("4", "32"):
        monkeypatch.setenv("GLASMA_CG_WALK", chunk)
        s1, U1, E1, G1 = _fixed(N, bc, f, algorithm, 4)
        assert np.abs(G1 - G0).max() < 1e-12, (N, chunk)
        assert np.abs(U1 - U0).max() < 1e-12
        assert np.abs(E1 - E0).max() < 1e-12
        assert np.abs(s1 - s0).max() < 1e-12 * max(1.0, np.abs(s0).max())


@pytest.mark.parametrize("dims", [(5, 16, 16), (3, 20, 50), (7, 64, 25), (2, 7, 130), (9, 128, 6), (4, 100, 35)])
def test_strided_groups(dims):
    """Strided passes of short and odd lengths against numpy: 1e-12 of the largest value."""
    from soerenpragya3dglasma_amd import fft_host
    rng = np.random.default_rng(sum(dims))
    x = rng.normal(size=tuple(reversed(dims)) + (3,)) + 1j * rng.normal(size=tuple(reversed(dims)) + (3,))
    ref = np.fft.fftn(x, axes=(0, 1, 2))
    assert np.abs(fft_host(x, dims, 3, -1) - ref).max() < 1e-12 * np.abs(ref).max()
    assert np.abs(fft_host(ref, dims, 3, +1) / np.prod(dims) - x).max() < 1e-12 * np.abs(x).max()
