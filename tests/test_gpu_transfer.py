"""Field transfers in pieces by several workers: every field comes back bit for bit, over lattices of one piece, of many,
with partial tiles and pieces, and from two threads with a context each."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _round_trip(N, bc, seed, fail):
    from soerenpragya3dglasma_amd import Glasma
    r = np.random.RandomState(seed)
    lay = {"U": (3, 3, 3), "E": (3, 8), "Jp": (8,), "Jm": (8,), "JpS": (8,), "JmS": (8,)}
    f = {}
    for k, tail in lay.items():
        v = r.standard_normal((N[2] + 2, N[1], N[0]) + tail)
        f[k] = v + 1j * r.standard_normal(v.shape) if k == "U" else v
    with Glasma(N, (1.0, 1.0, 1.0), 0.25, bc) as g:
        for _ in range(2):
            g.set_fields(f["U"], f["E"], f["Jp"], f["Jm"], f["JpS"], f["JmS"])
            g.set_uold(f["U"])
            d = g.get_fields()
            d["UOld"] = g.get_uold()
            for k, v in d.items():
                want = f["U" if k == "UOld" else k]
                lo, hi = (want[-2], want[1]) if bc else (want[1], want[-2])
                if not (np.array_equal(v[1:-1], want[1:-1]) and np.array_equal(v[0], lo) and np.array_equal(v[-1], hi)):
                    fail.append((N, k))


@pytest.mark.parametrize("N,bc", [((1, 1, 1), 0), ((3, 5, 7), 1), ((64, 6, 6), 0), ((64, 19, 2), 0), ((33, 31, 40), 1), ((48, 48, 20), 0)])
def test_fields_round_trip(N, bc):
    fail = []
    _round_trip(N, bc, 3, fail)
    assert not fail


def test_two_threads():
    fail = []
    th = [threading.Thread(target=_round_trip, args=((40, 40, 24), k, k, fail)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not fail
