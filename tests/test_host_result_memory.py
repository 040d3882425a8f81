"""The pinned memory that records write their results to: none is pinned for a context that records nothing, contexts share
it, and records and gauge fixing do without where none can be had."""
from tests import fake_runtime

SHARED = """
N = (6, 6, 12)
contexts = [Glasma(N) for _ in range(5)]
batch = GlasmaBatch([(N, (1.0, 1.0, 1.0), 0.25)] * 12)
assert fake.fake_pins() == 0, "making contexts pinned %d times" % fake.fake_pins()
for g in contexts + batch.events:
    g.bulk_raw(), g.emt_profile(), g.gauss(), g.transverse_energy_map()
    g.coulomb_gauge_algorithm("jacobi", 1e-9, 2)
assert fake.fake_pins() == 1, fake.fake_pins()
batch.close()
for g in contexts:
    g.close()
assert fake.fake_pinned() == 64 << 10
for _ in range(3):
    with Glasma(N) as g:
        g.bulk_raw()
assert fake.fake_pins() == 1
assert _lib.lib().glasma_release_idle() == 0 and fake.fake_pinned() == 0
"""

NONE = """
fake.fake_pin_limit(0)
with Glasma((6, 6, 12)) as g:
    copies = fake.fake_copies()
    g.bulk_raw(), g.emt_profile(), g.gauss(), g.transverse_energy_map()
    assert fake.fake_copies() == copies + 4
    g.coulomb_gauge_algorithm("jacobi", 1e-9, 2)
    assert fake.fake_copies() == copies + 5
"""


def test_contexts_share_the_result_memory():
    fake_runtime.run(SHARED)


def test_records_without_pinned_memory():
    fake_runtime.run(NONE)
