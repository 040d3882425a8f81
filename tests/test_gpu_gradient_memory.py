"""The gradient with as many segments kept whole as the caller's limit holds."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsteps,ckpt", [(12, 2), (11, 2), (7, 3), (3, 4)])
def test_gradient_is_the_same_under_any_limit(nsteps, ckpt):
    """Energies bit for bit, gradients to 1e-12 of their largest entry (the final state's link cotangent is scattered with
    atomic adds, whose order varies)."""
    from soerenpragya3dglasma_amd import Glasma
    N = (8, 6, 12)
    xl, _ = O.draw_charges(4, N[0], N[1], 0.5, 0.5)
    z = np.arange(N[2])
    rho = (np.exp(-0.5 * ((z - 5) / 2.0) ** 2) / np.sqrt(2 * np.pi * 4.0))[:, None, None, None] * xl[None]
    mv = Glasma.mv_params(lam=1.65, meff=0.1, sigma_l=2.0, sigma_r=2.0, center_l=5, center_r=7)
    step = 1312 * N[0] * N[1] * N[2]
    with Glasma(N, (1.0, 1.0, 1.0), 0.25) as g:
        e0, g0 = g.slab_energy_gradient(mv, rho, nsteps, ckpt, 6, 3)
        for limit in (1, 3 * ckpt * step, 1 << 40, 0):
            g.set_gradient_memory(limit)
            for _ in range(2):
                e, gr = g.slab_energy_gradient(mv, rho, nsteps, ckpt, 6, 3)
                assert e == e0, limit
                assert np.abs(gr - g0).max() <= 1e-12 * np.abs(g0).max(), limit
