"""The step's two register budgets (two or three tiles resident per CU) against the oracle, on both sides of each line of
the rule: up to 512 tiles two, up to 768 three, up to 1024 two, beyond three; both row forms.  Tolerance 1e-12 absolute as
for the other step tests: fields of order one, three steps of a few hundred operations each.
"""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import fields_maxdiff, random_fields, upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [(32, 32, 32), (32, 32, 33), (32, 32, 48), (32, 32, 49), (32, 32, 64), (32, 32, 65),
                               (40, 40, 20), (40, 40, 30), (40, 41, 33), (40, 40, 45)])
def test_step_residency(N):
    from soerenpragya3dglasma_amd import Glasma
    a, dt = (1.0, 0.85, 0.6), 0.1
    f = random_fields(N, seed=sum(N), bc=1)
    with Glasma(N, a, dt, 1) as g:
        upload(g, f)
        g.Update(3)
        d = g.get_fields()
        uold = g.get_uold()
    O.update(f, a, dt, 3, 1)
    diff = fields_maxdiff(d, f)
    print(N, diff)
    assert max(diff.values()) < 1e-12, (N, diff)
    assert np.abs(uold - f.UOld).max() < 1e-12
