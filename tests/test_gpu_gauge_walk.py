"""The z-walking deviation kernel against the other one on planes of several units with a ragged last one, with the walk
known to have been taken (test_cg_walk_plan.plan): one chunk and several, a short last chunk, both z boundaries, sites whose
neighbours lie in another unit.  Tolerance 1e-12, as for planes of one unit (test_gpu_gauge_shapes): the same sums, grouped
differently, a few hundred roundings of order-one terms."""
import numpy as np
import pytest

from tests.helpers import random_fields
from tests.test_cg_walk_plan import plan
from tests.test_gpu_gauge_shapes import _fixed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("algorithm,N,bc", [("jacobi", (31, 33, 5), 0), ("jacobi", (31, 33, 5), 1),
                                            ("jacobi", (25, 40, 6), 0), ("consistent", (25, 40, 6), 0),
                                            ("consistent", (25, 40, 6), 1), ("consistent", (100, 5, 9), 0),
                                            ("jacobi", (100, 5, 9), 1), ("consistent", (35, 36, 7), 1)])
def test_ragged_planes_of_several_units(monkeypatch, algorithm, N, bc):
    f = random_fields(N, seed=sum(N), link_scale=0.2, bc=bc)
    monkeypatch.setenv("GLASMA_CG_WALK", "0")
    s0, U0, E0, G0 = _fixed(N, bc, f, algorithm, 4)
    for chunk in (4, 32):
        zc, n = plan(N, 0, chunk)
        assert zc == chunk and n > (N[2] + chunk - 1) // chunk and N[0] * N[1] % 256  # taken, several units, ragged
        monkeypatch.setenv("GLASMA_CG_WALK", str(chunk))
        s1, U1, E1, G1 = _fixed(N, bc, f, algorithm, 4)
        assert np.abs(G1 - G0).max() < 1e-12, chunk
        assert np.abs(U1 - U0).max() < 1e-12
        assert np.abs(E1 - E0).max() < 1e-12
        assert np.abs(s1 - s0).max() < 1e-12 * max(1.0, np.abs(s0).max())
