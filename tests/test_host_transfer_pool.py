"""What a field transfer takes from the runtime: streams and pinned memory that the next context finds again, and no more
workers than buffers can be pinned."""
from tests import fake_runtime

CYCLES = """
N = (16, 16, 32)


def event():
    with Glasma(N) as g:
        before = fake.fake_streams(), fake.fake_pins()
        g.set_fields(**g.get_fields())
        return fake.fake_streams() - before[0], fake.fake_pins() - before[1]


event()
left = fake.fake_pinned()
assert left <= 8 << 20, left  # one set after the last context
for _ in range(5):
    assert event() == (0, 0), "a later context made streams or pinned memory again"
assert fake.fake_pinned() == left
assert _lib.lib().glasma_release_idle() == 0 and fake.fake_pinned() == 0
event()
"""

THREADS = """
import threading
N = (16, 16, 32)
ctx = [Glasma(N) for _ in range(6)]
f = [g.get_fields() for g in ctx]
wait = threading.Barrier(6)


def work(g, f):
    for _ in range(20):
        wait.wait()
        g.set_fields(**f)


th = [threading.Thread(target=work, args=a) for a in zip(ctx, f)]
held = fake.fake_pinned()
for t in th:
    t.start()
for t in th:
    t.join()
assert fake.fake_pins() <= 6 * 8 + 6 + 8, "sets were given up between the transfers of six threads"
for g in ctx:
    g.close()
assert fake.fake_pinned() <= 8 << 20
"""

SCARCE = """
N = (16, 16, 32)
with Glasma(N) as g:
    fake.fake_pin_limit(fake.fake_pinned() + (5 << 19))
    f = g.get_fields()
    g.set_fields(**f)
    fake.fake_pin_limit(1 << 30)
    g.set_fields(**f)
"""


def test_contexts_one_after_another_pin_once():
    fake_runtime.run(CYCLES)


def test_threads_keep_their_sets():
    fake_runtime.run(THREADS)


def test_fewer_workers_where_little_can_be_pinned():
    fake_runtime.run(SCARCE)
