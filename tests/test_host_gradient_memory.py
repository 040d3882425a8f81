"""The device memory that a gradient call leaves in its context: bounded by ckpt unless the caller allows more, given back
when asked."""
from tests import fake_runtime

SCRIPT = """
N, steps, ckpt = (8, 8, 16), 60, 2
S = N[0] * N[1] * N[2]
xl, _ = Glasma.draw_charges(1, N[0], N[1], 0.5, 0.5)
mv = Glasma.mv_params(1.65, 0.1, 2.0, 2.0, 5, 9)
rho = np.zeros((N[2], N[1], N[0], 8))
g = Glasma(N)


def held():
    b = ctypes.c_size_t()
    assert _lib.lib().glasma_memory_bytes(g._h, ctypes.byref(b)) == 0
    return b.value


empty, empty_device = held(), fake.fake_used()


def after(nbytes=None):
    if nbytes is not None:
        g.set_gradient_memory(nbytes)
    g.slab_energy_gradient(mv, rho, steps, ckpt, 8, 4)
    return held() - empty


def bound(sets):  # the sets, a checkpoint of 110 planes per segment, and the cotangents and sheets of a call
    return 8 * S * (sets * ckpt * 164 + (steps // ckpt + 1) * 110 + 700)


every = 1 << 40
print(after(), bound(2))
assert after() <= bound(2)
assert after(every) >= 8 * S * steps * 164  # all thirty segments
assert after(5 * ckpt * 1312 * S) <= bound(5)
assert after(1) <= bound(1)
assert after(every) >= 8 * S * steps * 164
fft = 2 * 16 * S * 8  # the transforms' work array and the reductions stay
g.set_gradient_memory(0)
assert held() - empty <= fft and fake.fake_used() - empty_device <= fft, (held() - empty, fake.fake_used() - empty_device)
assert after() <= bound(2)
g.close()
"""


def test_gradient_memory_follows_ckpt():
    fake_runtime.run(SCRIPT)


FALLBACK = """
N, steps, ckpt = (8, 8, 16), 40, 2
S = N[0] * N[1] * N[2]
xl, _ = Glasma.draw_charges(1, N[0], N[1], 0.5, 0.5)
mv = Glasma.mv_params(1.65, 0.1, 2.0, 2.0, 5, 9)
rho = np.zeros((N[2], N[1], N[0], 8))
g = Glasma(N)
for message in (False, True):
    if message:  # a message that an earlier call left
        assert _lib.lib().glasma_set_wilson_lines(g._h, b"X", ctypes.byref(mv), None, None, None) != 0
    before = _lib.lib().glasma_last_error(g._h)
    assert bool(before) == message
    g.slab_energy_gradient(mv, rho, steps, ckpt, 8, 4)
    need = fake.fake_used()  # with two sets
    g.set_gradient_memory(1 << 40)
    fake.fake_show(288 << 30)
    fake.fake_limit(need + 8 * S * 3 * ckpt * 164)  # three sets more, though the device seems to have room for all
    for _ in range(2):
        g.slab_energy_gradient(mv, rho, steps, ckpt, 8, 4)
        assert _lib.lib().glasma_last_error(g._h) == before, _lib.lib().glasma_last_error(g._h)
        assert fake.fake_used() <= need
    g.set_gradient_memory(0)
    fake.fake_limit(need // 2)  # not even the two sets: an error
    try:
        g.slab_energy_gradient(mv, rho, steps, ckpt, 8, 4)
    except GlasmaError as e:
        assert "allocation" in str(e)
    else:
        raise SystemExit("no error")
    fake.fake_limit(288 << 30)
    fake.fake_show(0)
    g.close()
    g = Glasma(N)
"""


def test_fallback_to_two_sets_leaves_no_message():
    """When another user of the device takes the memory that seemed free, the call goes on with two sets, and
    glasma_last_error keeps what it said before."""
    fake_runtime.run(FALLBACK)
