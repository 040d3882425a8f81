"""MV initial states at the edges of the sheet kernels' sizes, against the oracle: odd and prime lengths, planes beyond
the LDS (the transverse factor in separate passes), z lines taken four, two and one at a time, one z layer (where the
two sheets' ranges overlap).

Tolerance 1e-11 of the largest |E| or |J|: the oracle's Wilson line is a product of up to Nz exponentials, each within
a few 1e-16, so up to 2048 * 4e-16 = 8e-13 at Nz = 2048, and E divides the logarithm of a product of two links by
dt = 0.25 (a factor 4); J is J-stat through factors of modulus <= 1.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("driver,N", [(0, (11, 13, 9)), (1, (72, 75, 3)), (0, (72, 75, 4)), (2, (4, 3, 600)),
                                      (0, (3, 5, 2048)), (0, (5, 7, 1)), (2, (1, 6, 10)), (0, (64, 64, 6)), (1, (56, 88, 4))])
def test_sheet_shapes(driver, N):
    from soerenpragya3dglasma_amd import Glasma
    a, dt = (1.0, 0.9, 1.1), 0.25
    kw = dict(lam=1.65, meff=0.1, sigma_l=2.0, sigma_r=2.5, center_l=N[2] // 3, center_r=N[2] // 2)
    xl, xr = O.draw_charges(5, N[0], N[1], 0.5, 0.5)
    f = O.mv_initial_state(driver, N, a, dt, xl, xr, **kw)
    with Glasma(N, a, dt, 0) as g:
        g.mv_initial_state(driver, Glasma.mv_params(mult_l=1.0, mult_r=1.0, **kw), xl, xr)
        d = g.get_fields()
        uold = g.get_uold()
    errs = {k: float(np.abs(d[k][1:-1] - getattr(f, k)[1:-1]).max()) for k in ("U", "E", "Jp", "Jm", "JpS", "JmS")}
    errs["UOld"] = float(np.abs(uold[1:-1] - f.UOld[1:-1]).max())
    scale = max(np.abs(f.E).max(), np.abs(f.JpS).max(), np.abs(f.JmS).max(), 1.0)
    print(driver, N, errs, scale)
    assert max(errs.values()) < 1e-11 * scale, errs


@pytest.mark.parametrize("D", ["L", "R"])
@pytest.mark.parametrize("N", [(9, 11, 1), (8, 8, 7), (5, 13, 65), (3, 50, 16), (128, 130, 4)])
def test_wilson_lines_in_runs(N, D):
    """The path-ordered product in runs along z, Nz below, at and past multiples of the number of runs and planes that do
    not fill their waves, against the oracle: V to 1e-12 (65 exponentials of a few 1e-16 each)."""
    from soerenpragya3dglasma_amd import Glasma
    a = (1.0, 0.9, 1.1)
    kw = dict(lam=1.65, meff=0.1, sigma_l=2.0, sigma_r=2.0, center_l=N[2] // 3, center_r=N[2] // 2)
    xl, _ = O.draw_charges(7, N[0], N[1], 0.6, 0.6)
    with Glasma(N, a, 0.25, 0) as g:
        V, _ = g.set_wilson_lines(D, Glasma.mv_params(mult_l=1.0, mult_r=1.0, **kw), xl)
    rho_old = np.zeros((N[2] + 2, N[1], N[0], 8))
    rho_o, V_o = np.zeros_like(rho_old), np.zeros((N[2] + 2, N[1], N[0], 3, 3), complex)
    V_o[..., 0, 0] = V_o[..., 1, 1] = V_o[..., 2, 2] = 1
    O.lib().ref_set_wilson_lines(O.ivec(N), O.dvec(a), 0, kw["lam"], kw["meff"], kw["sigma_l"], 1.0, O.P(xl), D.encode(),
                                 kw["center_l"] if D == "L" else kw["center_r"], O.P(rho_old), O.P(rho_o), O.P(V_o))
    assert np.abs(V[1:-1] - V_o[1:-1]).max() < 1e-12
