"""Charge gradient on a lattice whose blocks are no multiple of the eight XCD ranges of the backward passes.

18 x 14 x 33 has 33 site blocks (the last half full) and 99 (block, direction) units.  Tolerance 1e-6 as for the
smaller lattices: the Richardson difference of step 1e-3 leaves an O(1e-12) truncation and a round-off of about
1e-13 |E| / 1e-3 of the energy's scale.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def test_gradient_ragged_blocks():
    from soerenpragya3dglasma_amd import Glasma
    N = (18, 14, 33)
    xl, _ = O.draw_charges(3, N[0], N[1], 0.5, 0.5)
    z = np.arange(N[2])
    rho = (np.exp(-0.5 * ((z - 13) / 3.0) ** 2) / np.sqrt(2 * np.pi * 9.0))[:, None, None, None] * xl[None]
    mv = Glasma.mv_params(lam=1.65, meff=0.1, sigma_l=3.0, sigma_r=3.0, center_l=13, center_r=18)
    rng = np.random.default_rng(11)
    with Glasma(N, (1.0, 1.0, 1.0), 0.25) as g:
        _, grad = g.slab_energy_gradient(mv, rho, 4, 3, 17, 6)

        def cd(v, eps):
            return (g.slab_energy_from_charge(mv, rho + eps * v, 4, 17, 6) -
                    g.slab_energy_from_charge(mv, rho - eps * v, 4, 17, 6)) / (2 * eps)
        worst = 0.0
        for _ in range(6):
            v = rng.normal(size=rho.shape) * np.abs(rho).max()
            ad = float(np.sum(grad * v))
            worst = max(worst, abs((4.0 * cd(v, 5e-4) - cd(v, 1e-3)) / 3.0 - ad) / abs(ad))
    print(worst)
    assert worst < 1e-6


@pytest.mark.parametrize("nsteps,ckpt", [(12, 2), (11, 2), (7, 3)])
def test_gradient_any_number_of_segment_sets(monkeypatch, nsteps, ckpt):
    """One to all of the segments kept by the forward run, the rest recomputed: energies bit for bit, gradients to 1e-12
    of their largest entry (the final state's atomic scatter, as for the test of one and two sets)."""
    from soerenpragya3dglasma_amd import Glasma
    N = (8, 6, 12)
    xl, _ = O.draw_charges(4, N[0], N[1], 0.5, 0.5)
    z = np.arange(N[2])
    rho = (np.exp(-0.5 * ((z - 5) / 2.0) ** 2) / np.sqrt(2 * np.pi * 4.0))[:, None, None, None] * xl[None]
    mv = Glasma.mv_params(lam=1.65, meff=0.1, sigma_l=2.0, sigma_r=2.0, center_l=5, center_r=7)
    monkeypatch.setenv("GLASMA_GRAD_SETS", "1")
    with Glasma(N, (1.0, 1.0, 1.0), 0.25) as g:
        e1, g1 = g.slab_energy_gradient(mv, rho, nsteps, ckpt, 6, 3)
        for sets in ("2", "3", "5", None):  # the same context: its arrays change their places
            monkeypatch.setenv("GLASMA_GRAD_SETS", sets) if sets else monkeypatch.delenv("GLASMA_GRAD_SETS")
            for _ in range(2):
                e, gr = g.slab_energy_gradient(mv, rho, nsteps, ckpt, 6, 3)
                assert e == e1, sets
                assert np.abs(gr - g1).max() <= 1e-12 * np.abs(g1).max(), sets
