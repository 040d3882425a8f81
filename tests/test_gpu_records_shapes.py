"""The records' block shapes: layers per thread of the transverse map (1 and more), partial last chunks and plane chunks,
and per-layer sums over more than 64 blocks, against numpy on the fields copied out of the context.  Every entry is a sum
of positive terms of order one formed to a few units of the last place, so entries agree to far better than 1e-12 of
themselves."""
import numpy as np
import pytest

from tests.helpers import random_fields, site_fields_np, upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,bc", [((5, 3, 2), 0), ((16, 16, 33), 1), ((48, 48, 130), 0), ((130, 131, 3), 1), ((129, 128, 5), 0)])
def test_records_match_numpy(N, bc):
    from soerenpragya3dglasma_amd import Glasma
    a = (1.0, 0.9, 0.8)
    f = random_fields(N, seed=3, bc=bc)
    with Glasma(N, a, 0.2, bc) as g:
        upload(g, f)
        bulk, prof, emap = g.bulk_raw(), g.field_profile(), g.transverse_energy_map()
    E2, B = site_fields_np(f)
    want = np.concatenate([E2.sum((0, 1, 2)), B.sum((0, 1, 2)), [0, 0]])
    assert np.abs(bulk[:8] - want).max() <= 1e-12 * np.abs(want).max()
    src = (f.E[1:-1, ..., 2, :] * (f.Jp - f.Jm)[1:-1]).sum() / np.sqrt(2.0)
    assert abs(bulk[8] - src) <= 1e-12 * np.abs(f.E[1:-1, ..., 2, :] * (f.Jp - f.Jm)[1:-1]).sum()
    e, b = E2.mean((1, 2)), B.mean((1, 2))
    cols = 0.5 * np.stack([b[:, 0] + b[:, 1], b[:, 2], e[:, 0] + e[:, 1], e[:, 2]], -1)
    assert np.abs(prof - cols).max() <= 1e-12 * np.abs(cols).max()
    c = (np.array(a) / np.prod(a)) ** 2
    t = 0.5 * ((E2 + B) * c).sum(-1) / N[2]
    cut = (N[2] - 2) // 2 + 1
    want = np.stack([t[:cut].sum(0), t[cut:].sum(0)], -1)
    assert np.abs(emap - want).max() <= 1e-12 * np.abs(want).max()
