"""A kernel launch that the runtime refuses ends its call with an error, whichever of the call's launches it is: no result
of an earlier call is returned in its place, and no error is left for the next call."""
import pytest

from tests import fake_runtime

SCRIPT = """
N = (6, 10, 12)
xl, xr = Glasma.draw_charges(1, N[0], N[1], 0.5, 0.5)
mv = Glasma.mv_params(1.65, 0.1, 2.0, 2.0, 4, 7)
rho = np.zeros((N[2], N[1], N[0], 8))
g = Glasma(N)
calls = {{
    "records": [g.bulk_raw, g.gauss, g.unitarity, g.emt_profile, g.field_profile, g.current_profile,
                g.transverse_energy_map, g.checksum],
    "fields": [g.get_fields, lambda: g.set_fields(**g.get_fields()), g.get_uold, g.get_gauge_fixed],
    "gauge": [lambda: g.coulomb_gauge(1e-9, 3), lambda: g.coulomb_gauge_algorithm("consistent", 1e-9, 3),
              lambda: g.coulomb_gauge_algorithm("jacobi", 1e-9, 3), g.gauss_restore],
    "states": [lambda: g.mv_initial_state(0, mv, xl, xr), lambda: g.set_wilson_lines("L", mv, xl),
               lambda: g.slab_energy(6, 3), lambda: g.slab_energy_from_charge(mv, rho, 3, 6, 3),
               lambda: g.slab_energy_gradient(mv, rho, 5, 2, 6, 3)],
}}[{which!r}]
g.coulomb_gauge(1e-9, 1)
g.Update(1)
for call in calls:
    call()  # what a first call prepares is there
    n = fake.fake_launches()
    call()
    n = fake.fake_launches() - n
    for k in range(n):
        fake.fake_refuse_launch(k)
        try:
            call()
        except GlasmaError:
            pass
        else:
            raise SystemExit("launch %d of %d refused, and no error from %r" % (k, n, call))
        fake.fake_refuse_launch(-1)
        call()
    print(n)
"""


@pytest.mark.parametrize("which", ["records", "fields", "gauge", "states"])
def test_refused_launch_is_an_error(which):
    assert all(int(n) > 0 for n in fake_runtime.run(SCRIPT.format(which=which)).split())
