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
